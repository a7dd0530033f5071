// 2-D convolution / local filtering and average pooling of one image signal.
//
// Convolution: a group owns a tile of output pixels x a tile of filters.  For one
// chunk of input channels at a time it stages the input patch under its pixels and
// the taps of its filters in LDS, then every thread accumulates its (pixel, filter)
// output over the chunk's channels and the kernel taps from LDS alone.  The accumulation order per output element is
// channel, kernel row, kernel column, one fused multiply-add each, as in the loop
// of clra_nonlinearities.py:1812-1845; channel chunks are visited in order, so
// chunking does not change it.  With channels last the filter index runs fastest
// over the lanes (filter taps and output stores coalesce, patch reads broadcast);
// with channels first the pixel column does.
// What happens to an output besides being stored (the epilogues of the products): the filters that it
// feeds are stepped, or the current it drives is formed and the neuron updated.  Launches of their
// own for either cost 4-5 us of a step each: whole steps of two layers of filters over 28 x 28 pixels
// 39.0 us -> 26.3, 40 x 40 x 3 pixels 47.6 -> 33.6, 48 x 48 x 3 92.2 -> 81.4.
#include <cstring>
#include <type_traits>

#include "nhip_common.h"
#include "neuron_math.h"

namespace {

#define NHIP_STREAM(s) static_cast<hipStream_t>(s)

constexpr int STAGE_PF = 8;   // loads in flight per lane while staging the patch
constexpr int FILT_PF = 16;   // ... and the filter taps

struct ConvGeom {
    int nxi, nxj, nc, nyi, nyj, nf;
    int si, sj, sti, stj, pi, pj;
    int xs_i, xs_j, xs_c, ys_i, ys_j, ys_f;
    int x_start, y_start, f_start;
    int tile_i, tile_j, tile_f, c_chunk, local, f_fast;
    int nipatch, njpatch, tiles_j;
};

struct ConvEpi {
    EpilogueArgs args;       // filters: targets 0 .. n_targets; neurons: population 0
    int n_targets;
    // current of output i: beta * yin + alpha * (a * A[x_start]) + gamma, the sums of a product with one
    // column (or none: a_start CONV_NONE); yin and a are elements of A, or the output (CONV_OUT)
    const float* A;
    float* J;
    int a_start, a_stride0, x_start, j_start;  // j_start < 0: the current is not stored
    float alpha, beta, gamma;
    int yin_start, yin_stride0;
};
constexpr int CONV_NONE = -1, CONV_OUT = -2;

// What the epilogue of output i needs from memory, requested before the sum is formed (after it:
// 28 x 28 pixels 26.3 us a step instead of 26.1, 48 x 48 x 3 pixels 81.4 instead of 80.7).
struct ConvAhead {
    FilterTarget target;
    LifPop pop;
    NeuronPop npop;
    float f, v, w, n, yin, a, x;
};

template <int EPI>
__device__ __forceinline__ ConvAhead conv_ahead(const ConvEpi& e, int i) {
    ConvAhead r = {};
    if (epi_filters(EPI)) {
        r.target = e.args.filter.targets[0];
        r.f = e.args.filter.F[(size_t)r.target.y_start + i];
    }
    if (EPI != EPI_LIF && EPI != EPI_NEURON) return r;
    const LifArgs& a = e.args.lif;
    if (EPI == EPI_LIF) {
        r.pop = a.pops[0];
        r.v = a.V[(size_t)r.pop.v_start + i];
        r.w = a.W[(size_t)r.pop.w_start + i];
    } else {
        r.npop = *reinterpret_cast<const NeuronPop*>(a.pops);
        if (neuron_has_v(r.npop.kind)) r.v = a.V[(size_t)r.npop.v_start + i];
        if (neuron_has_w(r.npop.kind)) r.w = a.W[(size_t)r.npop.w_start + i];
        if (neuron_has_n(r.npop.kind)) r.n = a.N[(size_t)r.npop.n_start + i];
    }
    if (e.yin_start != CONV_OUT) r.yin = e.A[e.yin_start + (size_t)i * e.yin_stride0];
    if (e.a_start != CONV_NONE) {
        r.x = e.A[e.x_start];
        if (e.a_start != CONV_OUT) r.a = e.A[e.a_start + (size_t)i * e.a_stride0];
    }
    return r;
}

template <int EPI>
__device__ __forceinline__ void conv_finish(const ConvEpi& e, const ConvAhead& r, int i, float out) {
    if (epi_filters(EPI)) {
        constexpr bool SECOND = EPI == EPI_FILTER2;
        const FilterArgs& f = e.args.filter;
        f.F[(size_t)r.target.y_start + i] = filter_step<SECOND>(f.targets, r.target, i, out, r.f);
        filter_epilogue<SECOND>(f, make_int2(1, e.n_targets - 1), i, out);
    }
    if (EPI != EPI_LIF && EPI != EPI_NEURON) return;
    float sum = e.beta * (e.yin_start == CONV_OUT ? out : r.yin);
    if (e.a_start != CONV_NONE) {
        const float p = fmaf(e.a_start == CONV_OUT ? out : r.a, r.x, 0.0f);
        sum = sum + e.alpha * ((p + 0.0f) + (0.0f + 0.0f));
    }
    const float j = sum + e.gamma;
    if (e.j_start >= 0) e.J[(size_t)e.j_start + i] = j;
    if (EPI == EPI_LIF) lif_epilogue(e.args.lif, r.pop, i, j, r.v, r.w);
    if (EPI == EPI_NEURON) neuron_epilogue(e.args.lif, r.npop, i, j, r.v, r.w, r.n);
}

template <int EPI>
__global__ __launch_bounds__(NHIP_WG) void conv2d_kernel(const ConvGeom g, const float* X,
                                                         const float* F, float* Y, const ConvEpi epi) {
    // [c_chunk][nipatch][njpatch] input patch, then (convolution only) the filter taps
    // of the group's filters [taps][channels of the chunk][tile_f], then the patch offset
    // of every tap
    extern __shared__ float lds[];
    const int tid = threadIdx.x;
    const int tile = blockIdx.x;
    const int i_base = (tile / g.tiles_j) * g.tile_i;
    const int j_base = (tile % g.tiles_j) * g.tile_j;
    const int k_base = blockIdx.y * g.tile_f;
    const int npatch = g.nipatch * g.njpatch;
    const int taps = g.si * g.sj;
    float* patch = lds;
    float* filt = patch + g.c_chunk * npatch;
    int* tap_off = reinterpret_cast<int*>(filt + (g.local ? 0 : g.c_chunk * taps * g.tile_f));

    const int n_pix = g.tile_i * g.tile_j;
    int pix, kf;
    if (g.f_fast) {
        kf = tid % g.tile_f;
        pix = tid / g.tile_f;
    } else {
        pix = tid % n_pix;
        kf = tid / n_pix;
    }
    const int ti = pix / g.tile_j, tj = pix - ti * g.tile_j;
    const int i = i_base + ti, j = j_base + tj, k = k_base + kf;
    const bool active = (pix < n_pix) && (kf < g.tile_f) && (i < g.nyi) && (j < g.nyj) &&
                        (k < g.nf);

    const int at = active ? k * g.ys_f + i * g.ys_i + j * g.ys_j : 0;
    const ConvAhead ahead = conv_ahead<EPI>(epi, at);

    const int i0 = i_base * g.sti - g.pi;
    const int j0 = j_base * g.stj - g.pj;
    const float* x = X + g.x_start;
    const float* f = F + g.f_start;
    for (int tap = tid; tap < taps; tap += NHIP_WG)
        tap_off[tap] = (tap / g.sj) * g.njpatch + tap % g.sj;

    float out = 0.0f;
    for (int c0 = 0; c0 < g.nc; c0 += g.c_chunk) {
        const int cc = min(g.c_chunk, g.nc - c0);
        // staging: STAGE_PF independent global loads per lane are issued before the
        // first of them is stored (few groups run, so nothing else hides the latency)
        for (int base = tid; base < cc * npatch; base += NHIP_WG * STAGE_PF) {
            float v[STAGE_PF];
            int where[STAGE_PF];
#pragma unroll
            for (int u = 0; u < STAGE_PF; ++u) {
                const int idx = base + u * NHIP_WG;
                v[u] = 0.0f;
                where[u] = -1;
                if (idx < cc * npatch) {
                    int c, kij;
                    if (g.f_fast) {  // channels last: channel is the unit-stride axis of X
                        c = idx % cc;
                        kij = idx / cc;
                    } else {
                        kij = idx % npatch;
                        c = idx / npatch;
                    }
                    const int ki = kij / g.njpatch, kj = kij - ki * g.njpatch;
                    const int ii = i0 + ki, jj = j0 + kj;
                    where[u] = c * npatch + kij;
                    if (ii >= 0 && ii < g.nxi && jj >= 0 && jj < g.nxj)
                        v[u] = x[(size_t)(c0 + c) * g.xs_c + (size_t)ii * g.xs_i +
                                 (size_t)jj * g.xs_j];
                }
            }
#pragma unroll
            for (int u = 0; u < STAGE_PF; ++u)
                if (where[u] >= 0) patch[where[u]] = v[u];
        }
        if (!g.local) {
            // filters are (tap, channel, filter) in memory, filter index at unit stride;
            // the LDS copy is [tap][channel of the chunk][filter of the tile].  All loads
            // of a lane are in flight before the first is stored; tile_f is a power of two.
            const int lg_f = __ffs(g.tile_f) - 1;
            const int total = (taps * cc) << lg_f;
            const float inv_cc = __frcp_rn((float)cc);
            for (int base = tid; base < total; base += NHIP_WG * FILT_PF) {
                float v[FILT_PF];
#pragma unroll
                for (int u = 0; u < FILT_PF; ++u) {
                    const int idx = base + u * NHIP_WG;
                    v[u] = 0.0f;
                    if (idx < total) {
                        const int q = idx & (g.tile_f - 1), r = idx >> lg_f;  // r = tap * cc + c
                        int tap = (int)((float)r * inv_cc);
                        if ((tap + 1) * cc <= r) ++tap;
                        if (tap * cc > r) --tap;
                        const int c = r - tap * cc;
                        if (k_base + q < g.nf)
                            v[u] = f[((size_t)tap * g.nc + (c0 + c)) * g.nf + k_base + q];
                    }
                }
#pragma unroll
                for (int u = 0; u < FILT_PF; ++u)
                    if (base + u * NHIP_WG < total) filt[base + u * NHIP_WG] = v[u];
            }
        }
        __syncthreads();
        if (active) {
            const float* p = patch + (g.sti * ti) * g.njpatch + g.stj * tj;
            if (g.local) {
                for (int c = 0; c < cc; ++c)
                    for (int tap = 0; tap < taps; ++tap) {
                        const float w = f[((size_t)(k * g.nc + c0 + c) * taps + tap) *
                                              (g.nyi * g.nyj) + i * g.nyj + j];
                        out = fmaf(w, p[c * npatch + tap_off[tap]], out);
                    }
            } else {
                // A lane's output is one chain of fused multiply-adds in a fixed order, and
                // small problems leave one wave per SIMD: the LDS reads of up to four
                // taps of a kernel row are issued together, ahead of their chain links.
                const float* w = filt + kf;
                for (int c = 0; c < cc; ++c) {
                    for (int ii = 0; ii < g.si; ++ii) {
                        const float* pr = p + c * npatch + ii * g.njpatch;
                        const float* wr = w + (ii * g.sj * cc + c) * g.tile_f;
                        for (int jj = 0; jj < g.sj; jj += 4) {
                            // no branches between the loads: past the row's end the last
                            // tap is read again and its chain link discarded
                            float pv[4], wv[4];
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                const int jq = min(jj + q, g.sj - 1);
                                pv[q] = pr[jq];
                                wv[q] = wr[jq * cc * g.tile_f];
                            }
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                const float next = fmaf(wv[q], pv[q], out);
                                out = (jj + q < g.sj) ? next : out;
                            }
                        }
                    }
                }
            }
        }
        __syncthreads();
    }
    if (active) {
        Y[g.y_start + (size_t)at] = out;
        conv_finish<EPI>(epi, ahead, at, out);
    }
}

// The same convolution (channels last) for images with too few outputs to fill the device with
// the tiles above.  A group is one wave: 16 filters x 4 consecutive pixels, an output per lane,
// so a few thousand outputs spread over all compute units instead of sharing a few.  All taps
// of the 16 filters and the windows of the 4 pixels are staged at once, every load of a lane in
// flight before the first is stored (memory is about a microsecond away and little else is
// running), in the order the sum walks them: LDS reads of the chain have constant offsets
// and no address arithmetic.  Same order, channel, kernel row, kernel column, one fused
// multiply-add each; taps outside the image multiply a zero, as the padded patch above does.
// 26 x 26 x 32 -> 12 x 12 x 64 (9,216 outputs of 288 links) 28.4 -> 7.7 us, 46 x 46 x 40 -> 22 x 22 x 80
// 41.8 -> 13.0.  Bound by the one trip to memory and the chain; which launches take it: see
// `conv_takes_waves`.
constexpr int CONV_WF = 16, CONV_WP = 4;
constexpr int CONV_WAVE_PF = 24;          // loads in flight per lane
constexpr int CONV_WAVE_LINKS = 16;       // chain links whose operands are read together
constexpr int CONV_WAVE_MAX_LINKS = 800;  // 64,000 bytes of LDS
constexpr int CONV_WAVE_MIN_LINKS = 64;
constexpr long long CONV_WAVE_MAX_OUT = 1 << 20;
// ... resident groups of a launch: the LDS of 256 compute units, at most 8 waves per SIMD
constexpr int CONV_N_CU = 256, CONV_CU_LDS = 160 * 1024, CONV_CU_WAVES = 32;

// VEC: filters in whole aligned quads
template <bool VEC, int EPI>
__global__ __launch_bounds__(NHIP_WAVE) void conv2d_wave_kernel(
    const ConvGeom g, const float* __restrict__ X, const float* __restrict__ F, float* Y,
    const ConvEpi epi) {
    extern __shared__ float4 lds4[];
    const int lane = threadIdx.x;
    const int taps = g.si * g.sj, n_links = taps * g.nc, n_pix = g.nyi * g.nyj;
    const int k0 = blockIdx.y * CONV_WF, pix0 = blockIdx.x * CONV_WP;
    float* wl = reinterpret_cast<float*>(lds4);  // [link][filter]
    float* xl = wl + n_links * CONV_WF;          // [link][pixel]
    constexpr int PF = CONV_WAVE_PF;
    const int kf = lane & (CONV_WF - 1), p = lane / CONV_WF;
    const bool active = k0 + kf < g.nf && pix0 + p < n_pix;
    const int at = active ? (pix0 + p) * g.nf + k0 + kf : 0;
    const ConvAhead ahead = conv_ahead<EPI>(epi, at);
    {   // taps: memory order is (tap, channel, filter)
        const float inv_nc = __frcp_rn((float)g.nc);
        constexpr int PER = VEC ? 4 : 1, LANES = CONV_WF / PER, ROWS = NHIP_WAVE / LANES;
        const int q = PER * (lane % LANES), row = lane / LANES;
        const float* f = F + g.f_start + k0;
        const int qc = min(q, max(g.nf - k0 - PER, 0));  // (filters past the last are not stored)
#pragma unroll 1
        for (int m0 = row; m0 < n_links; m0 += ROWS * PF) {
            float v[PF][PER];
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                const float* src = f + (size_t)min(m0 + u * ROWS, n_links - 1) * g.nf + qc;
                if (VEC) {
                    const float4 t = *reinterpret_cast<const float4*>(src);
                    v[u][0] = t.x; v[u][PER > 1 ? 1 : 0] = t.y;
                    v[u][PER > 1 ? 2 : 0] = t.z; v[u][PER > 1 ? 3 : 0] = t.w;
                } else {
                    v[u][0] = *src;
                }
            }
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                const int m = m0 + u * ROWS;
                int tap = (int)((float)m * inv_nc);  // m < 800: exact after one correction
                if ((tap + 1) * g.nc <= m) ++tap;
                if (tap * g.nc > m) --tap;
                const int e = (m - tap * g.nc) * taps + tap;
                if (m < n_links) {
#pragma unroll
                    for (int p = 0; p < PER; ++p) wl[e * CONV_WF + q + p] = v[u][p];
                }
            }
        }
    }
    {   // windows: 16 lanes per pixel, each a channel of 16; (tap, run of 16 channels) in turn
        const int p = lane >> 4, cl = lane & 15;
        const int pix = min(pix0 + p, n_pix - 1);
        const int i = pix / g.nyj, j = pix - i * g.nyj;
        const int i0 = i * g.sti - g.pi, j0 = j * g.stj - g.pj;
        const float* x = X + g.x_start;
        const int runs = (g.nc + 15) >> 4, n_loads = taps * runs;
        int t_i = 0, t_j = 0, run = 0;  // of the next load, the same for all lanes
#pragma unroll 1
        for (int l0 = 0; l0 < n_loads; l0 += PF) {
            float v[PF];
            int where[PF];
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                const int c = 16 * run + cl, ii = i0 + t_i, jj = j0 + t_j;
                const bool in = (unsigned)ii < (unsigned)g.nxi && (unsigned)jj < (unsigned)g.nxj;
                where[u] = (l0 + u < n_loads && c < g.nc)
                               ? (c * taps + t_i * g.sj + t_j) * CONV_WP + p : -1;
                const float t = x[in ? (ii * g.nxj + jj) * g.nc + min(c, g.nc - 1) : 0];
                v[u] = in ? t : 0.0f;
                ++run;
                const bool next_tap = run == runs;
                run = next_tap ? 0 : run;
                t_j += next_tap ? 1 : 0;
                const bool next_row = t_j == g.sj;
                t_j = next_row ? 0 : t_j;
                t_i += next_row ? 1 : 0;
            }
#pragma unroll
            for (int u = 0; u < PF; ++u)
                if (where[u] >= 0) xl[where[u]] = v[u];
        }
    }
    __syncthreads();
    const float* wp = wl + kf;
    const float* xp = xl + p;
    constexpr int U = CONV_WAVE_LINKS;
    float out = 0.0f;
    float wa[U], xa[U], wb[U], xb[U];
    auto read = [&](float (&w)[U], float (&x)[U], int e) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            w[u] = wp[(e + u) * CONV_WF];
            x[u] = xp[(e + u) * CONV_WP];
        }
    };
    auto sum = [&](const float (&w)[U], const float (&x)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) out = fmaf(w[u], x[u], out);
    };
    int e = 0;
    if (n_links >= U) {
        read(wa, xa, 0);
#pragma unroll 1
        for (; e + 3 * U <= n_links; e += 2 * U) {
            read(wb, xb, e + U);
            sum(wa, xa);
            read(wa, xa, e + 2 * U);
            sum(wb, xb);
        }
        sum(wa, xa);
        e += U;
    }
#pragma unroll 4
    for (; e < n_links; ++e) out = fmaf(wp[e * CONV_WF], xp[e * CONV_WP], out);
    if (active) {
        Y[g.y_start + (size_t)at] = out;
        conv_finish<EPI>(epi, ahead, at, out);
    }
}

struct PoolGeom {
    int nc, nyi, nyj, nxi, nxj, si, sj, sti, stj, x_start, y_start;
};

// Mean over the window's in-range, non-NaN inputs, summed row by row
// (clra_nonlinearities.py:2027-2041); channels first.
__global__ __launch_bounds__(NHIP_WG) void pool2d_kernel(const PoolGeom g, const float* X,
                                                         float* Y) {
    const int n = g.nc * g.nyi * g.nyj;
    const int e = blockIdx.x * NHIP_WG + threadIdx.x;
    if (e >= n) return;
    const int c = e / (g.nyi * g.nyj);
    const int ij = e - c * (g.nyi * g.nyj);
    const int i = ij / g.nyj, j = ij - i * g.nyj;
    const float* xc = X + g.x_start + (size_t)c * g.nxi * g.nxj;
    float out = 0.0f;
    int count = 0;
    for (int ii = 0; ii < g.si; ++ii) {
        for (int jj = 0; jj < g.sj; ++jj) {
            const int r = i * g.sti + ii, q = j * g.stj + jj;
            if (r < g.nxi && q < g.nxj) {
                const float v = xc[(size_t)r * g.nxj + q];
                if (!isnan(v)) {
                    out = __fadd_rn(out, v);
                    ++count;
                }
            }
        }
    }
    Y[g.y_start + e] = __fdiv_rn(out, (float)count);
}

// A group of one wave, or a tile?  A group's staging is paid per 4 pixels, a tile's per tile: the groups
// win while they are all resident at once, and lose in proportion to their rounds after that
// unless the tiles need several rounds too, or waste their lanes.  Measured (780 shapes, kernel time in
// us, groups / tiles; kernel, channels, filters; image sides 28, 64, 128, 256):
//   3 x 3, 32, 16      7.8/20.6    9.8/21.2   26.6/36.7    79.7/108.8
//   3 x 3, 32, 2      10.8/23.0   13.0/23.6   37.0/24.2   118.5/28.7
//   3 x 3, 32, 64      9.2/28.8   25.8/45.9   78.7/148.0       -
//   3 x 3, 88, 64     39.6/74.1  152.8/119.3       -           -
//   3 x 3,  8, 4       6.1/7.8     7.5/7.9    13.5/8.0     40.9/12.5
//   1 x 1, 200, 16        -        9.1/42.0        -       58.8/221.1   (no window to share in a tile)
//   5 x 5 by 2, 3, 16  9.3/7.7         (few channels: the windows load 16 of them side by side)
//   7 x 7 by 2, 16, 64, side 200   353.9/215.6
// By the rule below the launch is at most 5 % behind the tiles on those of several taps (of a
// single tap: two are, by 10 and 25 %), and 0.7 % behind the better of the two on average.
bool conv_takes_waves(const ConvGeom& g, long long n_tiles, long long n_groups) {
    const int taps = g.si * g.sj, links = taps * g.nc;
    if (!g.f_fast || g.local || (long long)g.nyi * g.nyj * g.nf > CONV_WAVE_MAX_OUT ||
        links < CONV_WAVE_MIN_LINKS || links > CONV_WAVE_MAX_LINKS)
        return false;
    const int lds = links * (CONV_WF + CONV_WP) * (int)sizeof(float);
    const long long resident = (long long)CONV_N_CU * min(CONV_CU_LDS / lds, CONV_CU_WAVES);
    // n_groups / resident <= rounds * max(1, n_tiles / tiles)
    auto within = [&](int rounds, int tiles) {
        return n_groups * tiles <= rounds * resident * max((long long)tiles, n_tiles);
    };
    if (taps == 1) return within(2, CONV_N_CU);
    if (g.nc < 8 || (links < 100 && n_groups > 2000)) return false;
    const bool cheap_groups = (g.nf >= 24 && !(g.nf & 3)) ||                 // taps in whole quads
                              (g.nc >= 32 && g.nf >= 4 && taps <= 9);       // full window loads
    return within(cheap_groups ? 2 : 1, 3 * CONV_N_CU);
}

// What a call with geometry `q` launches.
struct ConvLaunch {
    ConvGeom g;
    bool waves;  // conv2d_wave_kernel, else conv2d_kernel
    dim3 grid;
    int threads;
    size_t lds;
};

int conv_launch(const int* q, ConvLaunch& l) {
    ConvGeom& g = l.g;
    g.nxi = q[0]; g.nxj = q[1]; g.nc = q[2]; g.nyi = q[3]; g.nyj = q[4]; g.nf = q[5];
    g.si = q[6]; g.sj = q[7]; g.sti = q[8]; g.stj = q[9]; g.pi = q[10]; g.pj = q[11];
    g.x_start = q[12]; g.y_start = q[13]; g.f_start = q[14];
    const int channels_last = q[15];
    g.local = q[16];
    g.tile_i = q[17]; g.tile_j = q[18]; g.tile_f = q[19]; g.c_chunk = q[20];
    if (g.nxi <= 0 || g.nxj <= 0 || g.nc <= 0 || g.nyi <= 0 || g.nyj <= 0 || g.nf <= 0 ||
        g.si <= 0 || g.sj <= 0 || g.sti <= 0 || g.stj <= 0 || g.pi < 0 || g.pj < 0 ||
        g.x_start < 0 || g.y_start < 0 || g.f_start < 0)
        return NHIP_E_BADARG;
    if (g.tile_i <= 0 || g.tile_j <= 0 || g.tile_f <= 0 || g.c_chunk <= 0 ||
        (long long)g.tile_i * g.tile_j * g.tile_f > NHIP_WG)
        return NHIP_E_BADARG;
    g.f_fast = channels_last ? 1 : 0;
    g.xs_i = g.nxj * (channels_last ? g.nc : 1);
    g.xs_j = channels_last ? g.nc : 1;
    g.xs_c = channels_last ? 1 : g.nxi * g.nxj;
    g.ys_i = g.nyj * (channels_last ? g.nf : 1);
    g.ys_j = channels_last ? g.nf : 1;
    g.ys_f = channels_last ? 1 : g.nyi * g.nyj;
    g.nipatch = (g.tile_i - 1) * g.sti + g.si;
    g.njpatch = (g.tile_j - 1) * g.stj + g.sj;
    g.tiles_j = (g.nyj + g.tile_j - 1) / g.tile_j;
    const int tiles_i = (g.nyi + g.tile_i - 1) / g.tile_i;
    const size_t taps = (size_t)g.si * g.sj;
    l.lds = ((size_t)g.c_chunk * (g.nipatch * g.njpatch + (g.local ? 0 : taps * g.tile_f)) + taps) *
            sizeof(float);
    if (l.lds > 64 * 1024) return NHIP_E_BADARG;
    l.grid = dim3(g.tiles_j * tiles_i, (g.nf + g.tile_f - 1) / g.tile_f);
    l.threads = NHIP_WG;
    const dim3 waves((g.nyi * g.nyj + CONV_WP - 1) / CONV_WP, (g.nf + CONV_WF - 1) / CONV_WF);
    l.waves = conv_takes_waves(g, (long long)l.grid.x * l.grid.y, (long long)waves.x * waves.y);
    if (l.waves) {
        l.grid = waves;
        l.threads = NHIP_WAVE;
        l.lds = taps * g.nc * (CONV_WF + CONV_WP) * sizeof(float);
    }
    return 0;
}

}  // namespace

namespace {

template <int EPI>
int launch_conv(void* stream, const int* geom, const float* X, const float* F, float* Y, const ConvEpi& epi) {
    if (!geom || !X || !F || !Y) return NHIP_E_BADARG;
    ConvLaunch l;
    const int err = conv_launch(geom, l);
    if (err) return err;
    const ConvGeom& g = l.g;
    const dim3 block(l.threads);
    auto launch = [&](auto kernel) {
        NHIP_LAUNCH(kernel, l.grid, block, l.lds, NHIP_STREAM(stream), g, X, F, Y, epi);
    };
    if (!l.waves) launch(conv2d_kernel<EPI>);
    else if (!((g.nf | g.f_start) & 3) && !(reinterpret_cast<uintptr_t>(F) & 15)) launch(conv2d_wave_kernel<true, EPI>);
    else launch(conv2d_wave_kernel<false, EPI>);
    NHIP_LAUNCH_CHECK();
    return 0;
}

}  // namespace

extern "C" int nhip_conv2d(void* stream, const int* geom, const float* X, const float* F,
                           float* Y) {
    return launch_conv<EPI_NONE>(stream, geom, X, F, Y, ConvEpi{});
}

extern "C" int nhip_conv2d_filter(void* stream, const int* geom, const float* X, const float* F, float* Y,
                                  const int* targets, int n_targets, float* FO) {
    if (!targets || !FO || n_targets < 1) return NHIP_E_BADARG;
    ConvEpi epi{};
    epi.args.filter.targets = reinterpret_cast<const FilterTarget*>(targets);
    epi.args.filter.F = FO;
    epi.n_targets = n_targets;
    return launch_conv<EPI_FILTER2>(stream, geom, X, F, Y, epi);
}

extern "C" int nhip_conv2d_neuron(void* stream, const int* geom, const float* X, const float* F, float* Y,
                                  const float* A, const int* current, float* J, int lif, const int* pop,
                                  double dt, int upsample, float* V, float* W, float* S, float* N,
                                  const float* TAU, const float* REF, const float* AMP) {
    if (!A || !current || !J || !pop || !V || !W || !S || !N || upsample < 1 || !(dt > 0.0)) return NHIP_E_BADARG;
    ConvEpi epi{};
    epi.A = A;
    epi.J = J;
    epi.a_start = current[0];
    epi.a_stride0 = current[1];
    epi.x_start = current[2];
    epi.j_start = current[3];
    memcpy(&epi.alpha, current + 4, sizeof(float));
    memcpy(&epi.beta, current + 5, sizeof(float));
    memcpy(&epi.gamma, current + 6, sizeof(float));
    epi.yin_start = current[7];
    epi.yin_stride0 = current[8];
    if (epi.a_start < CONV_OUT || epi.yin_start < CONV_OUT || epi.yin_start == CONV_NONE || epi.x_start < 0)
        return NHIP_E_BADARG;
    LifArgs& a = epi.args.lif;
    a.pops = reinterpret_cast<const LifPop*>(pop);
    a.dt = (float)dt;
    a.dtu = (float)(dt / (double)upsample);  // formed in double and rounded once, as in nhip_lif
    a.dt_inv = (float)(1.0 / dt);
    a.upsample = upsample;
    a.V = V;
    a.W = W;
    a.S = S;
    a.N = N;
    a.TAU = TAU;
    a.REF = REF;
    a.AMP = AMP;
    return lif ? launch_conv<EPI_LIF>(stream, geom, X, F, Y, epi)
               : launch_conv<EPI_NEURON>(stream, geom, X, F, Y, epi);
}

extern "C" int nhip_conv2d_groups(const int* geom, int* n_groups, int* group_threads) {
    if (!geom || !n_groups || !group_threads) return NHIP_E_BADARG;
    ConvLaunch l;
    const int err = conv_launch(geom, l);
    if (err) return err;
    *n_groups = l.grid.x * l.grid.y;
    *group_threads = l.threads;
    return 0;
}

extern "C" int nhip_pool2d(void* stream, const int* geom, const float* X, float* Y) {
    if (!geom || !X || !Y) return NHIP_E_BADARG;
    PoolGeom g;
    g.nc = geom[0]; g.nyi = geom[1]; g.nyj = geom[2]; g.nxi = geom[3]; g.nxj = geom[4];
    g.si = geom[5]; g.sj = geom[6]; g.sti = geom[7]; g.stj = geom[8];
    g.x_start = geom[9]; g.y_start = geom[10];
    if (g.nc <= 0 || g.nyi <= 0 || g.nyj <= 0 || g.nxi <= 0 || g.nxj <= 0 || g.si <= 0 ||
        g.sj <= 0 || g.sti <= 0 || g.stj <= 0 || g.x_start < 0 || g.y_start < 0)
        return NHIP_E_BADARG;
    const long long n = (long long)g.nc * g.nyi * g.nyj;
    if (n > 0x7fffffffLL) return NHIP_E_BADARG;
    NHIP_LAUNCH(pool2d_kernel, dim3((unsigned)((n + NHIP_WG - 1) / NHIP_WG)),
                       dim3(NHIP_WG), 0, NHIP_STREAM(stream), g, X, Y);
    NHIP_LAUNCH_CHECK();
    return 0;
}
