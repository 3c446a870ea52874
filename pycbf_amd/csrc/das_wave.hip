// Launch of the wave-tile gather (das_wave.h) for nearest and linear, and the
// rules that pick it and its launch shape for every kind.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "das_wave.h"

namespace pycbf {

int wave_launch_sample(int gk, const DasArgs &a, const WaveArgs &w, int sum, int fc, int mode,
                       dim3 grid, int nw, size_t lds, hipStream_t s)
{
    if (gk == GK_NEAREST) return wave_sum<GK_NEAREST>(sum, fc, mode, a, w, grid, nw, lds, s);
    return wave_sum<GK_LINEAR>(sum, fc, mode, a, w, grid, nw, lds, s);
}

// Four frames of the gather table, the most that one pass reads.
static int64_t pass_table_bytes(const DasArgs &a)
{
    return (int64_t)a.ntx * a.nrx * a.ch_stride * 4 * 4;
}
constexpr int64_t BIG_TABLE = (int64_t)96 << 20;

// Whether each XCD takes every eighth outer element over all tiles, so that a
// channel's row enters one L2 only, instead of runs of tiles over all elements.
// Four or more frames; the outer axis has to give each of the 8 chunks two
// elements and more.  Times of this order over the other, and over the staged
// gather (k_das_lds):
//   tables over 96 MB per pass are pulled again by every XCD: 31 x 128 x 2048 x
//   200 x 200, k-order, 0.65 - 0.82, 60 x 64 x 2000, linear, 0.46 - 0.65;
//   smaller ones are not, and the chunks' partial images and idle waves cost
//   more: 16 x 48 x 800 onto 200 x 200, 16 frames, nearest 2.2 (1.36 of the
//   staged gather, the other 0.63), 12 x 128 x 1024, nearest, 2.1;
//   64 tiles and fewer leave the chip short of workgroups, of which this order has
//   8 times as many: 75 x 32 x 600 onto 1551 pixels, 4 frames, linear, 0.64.
// Images per element have no partials, and their chunks cost idle waves where
// the axis is short: 1 x 128 x 1024 onto 20 000 pixels, per transmit, 16
// frames, 4.9 of the other order (1.87 of the staged gather, the other 0.37).
static bool wave_slab(int gk, const DasArgs &a, int sum, int no, int ni, int64_t ntiles,
                      int64_t passes)
{
    const bool wide = gk == GK_KORDER || gk == GK_AKIMA;  // 16-byte entries
    const int64_t table = pass_table_bytes(a);
    // per-sample outputs: 0.4 - 1 over the geometry and a table beyond one L2, up to
    // 1.3 over delay tables (40 x 16 x 600, 16 frames), which each XCD reads whole
    if (sum == WS_NONE) return a.geo && ni >= 2 && no >= 16 && table >= (int64_t)4 << 20;
    const bool few = no >= 8 && ntiles * (wide ? 1 : passes) <= 64;
    const bool big = no >= 16 && table >= BIG_TABLE && (a.geo || no >= 48);
    if (sum == WS_BOTH) return few || big;
    if (ni == 1) return no >= 16 && passes >= 4 && ntiles > 64;
    if (few) return true;
    return wide ? no >= 16 : (a.sumflag == PYCBF_SUM_RX_ONLY ? no >= 32 : big);
}

bool das_wave_applies(int gk, const DasArgs &a)
{
    if (gk == GK_LINEAR && a.nsrc < 2) return false;      // reads pairs
    if (gk == GK_NEAREST && a.nsrc > 1 << 22) return false;  // nsrc - 1/2 as a float
    if (a.np > (int64_t)1 << 28) return false;  // 16 threads per pixel within a 32-bit grid
    // Nearest, sums of many transmits over many frames of a table beyond the L2s:
    // a sample is little more than its position, which the staged gather shares
    // among 16 frames and this one among 4 (16 frames of 75 x 40 x 3000 onto 128 x
    // 128: 474 us staged, 640 here; of 64 x 64 x 2000 onto 100 x 100: 376, 466).  At
    // 128 tiles and fewer, or few transmits, this one is faster all the same (31 x
    // 128 x 2048 onto 64 x 64: 0.56 of it).
    if (gk == GK_NEAREST && a.nfr > 8 && a.sumflag != PYCBF_SUM_NONE && a.ntx >= 50 &&
        a.np > 128 * 64 && pass_table_bytes(a) >= BIG_TABLE)
        return false;
    // the cubic over 4 or more frames is staged in LDS (k_das_cubic_dma)
    return gk != GK_CUBIC || a.nfr < 4;
}

// Length of the pixel grid's fast axis, read off two rows of delays (or of one
// coordinate, `stride` floats apart): along a line
// of pixels the delay to an element outside the line's span changes in one
// direction, and turns back where the next line starts.  The first turn of
// either row that divides the pixel count evenly is taken (the longer of the
// two, 0 when neither does).  Only the grouping of pixels into tiles depends
// on it, never a result.
constexpr int FAST_MIN = 32, FAST_MAX = 4096;

__global__ __launch_bounds__(1024) void k_fast_axis(const float *__restrict__ row0,
                                                    const float *__restrict__ row1, int stride,
                                                    int64_t np, int *__restrict__ fast)
{
    __shared__ int turn[2];
    if (threadIdx.x < 2) turn[threadIdx.x] = FAST_MAX;
    __syncthreads();
    const int n = (int)(np < FAST_MAX + 1 ? np : FAST_MAX + 1);
    float v[2][FAST_MAX / 1024][2];
    const float up[2] = {row0[stride] - row0[0], row1[stride] - row1[0]};
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int t = 0; t < FAST_MAX / 1024; ++t) {
            const int64_t p = (int64_t)min((int)threadIdx.x + t * 1024, n - 2) * stride;
            v[r][t][0] = (r ? row1 : row0)[p];
            v[r][t][1] = (r ? row1 : row0)[p + stride];
        }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        int first = FAST_MAX;
#pragma unroll
        for (int t = FAST_MAX / 1024 - 1; t >= 0; --t) {
            const int p = min((int)threadIdx.x + t * 1024, n - 2);
            if ((v[r][t][1] - v[r][t][0]) * up[r] < 0.0f) first = p + 1;
        }
        if (first < FAST_MAX) atomicMin(&turn[r], first);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int f = 0;
        for (int r = 0; r < 2; ++r)
            if (turn[r] >= FAST_MIN && turn[r] < FAST_MAX && turn[r] > f && np % turn[r] == 0)
                f = turn[r];
        *fast = f;
    }
}

int launch_fast_axis(const float *row0, const float *row1, int stride, int64_t np, int *fast,
                     hipStream_t s)
{
    hipLaunchKernelGGL(k_fast_axis, dim3(1), dim3(1024), 0, s, row0, row1, stride, np, fast);
    return check_launch("fast axis");
}

int launch_das_wave(int gk, const DasArgs &a0, int max_part, float *partial, int *fast,
                    hipStream_t s)
{
    DasArgs a = a0;
    WaveArgs w{};
    // pixels of unknown order over tables: patches of the grid they form
    // (images of some tiles only; a small one fits the caches in any order)
    if (a.geo == 0 && !a.perm && fast && a.np >= 4096) {
        const float *row = a.nrx >= 2 ? a.trx : a.ttx;
        const int64_t last = (a.nrx >= 2 ? a.nrx : a.ntx) - 1;
        if (int rc = launch_fast_axis(row, row + last * a.np, 1, a.np, fast, s)) return rc;
        w.fast = fast;
    }
    w.nhalf = (float)a.nsrc - 0.5f;
    const int sum = a.sumflag == PYCBF_SUM_TX_AND_RX ? WS_BOTH
                    : a.sumflag == PYCBF_SUM_NONE    ? WS_NONE
                                                     : WS_SEP;
    const int fc = a.nfr >= 4 ? 4 : (a.nfr >= 2 ? 2 : 1);
    const int mode = wave_mode_of(a.t0, a.dt, a.rdt, a.tmax, a.nsrc);
    w.weights = !(a.geo && a.thresh > 0.0f && a.thresh <= 1.0f);
    const int64_t ntiles = (a.np + 63) / 64;
    const int64_t passes = (a.nfr + fc - 1) / fc;
    // Waves per tile: the waves of a tile end together, so many small shares
    // leave more of them idle at its end, but few tiles need them to fill the
    // chip.  8 and 16 waves, us (cubic): 31 x 128 x 2048, 512 tiles 102 / 82, 1024
    // 128 / 118, 4096 360 / 346; 11 x 64 x 1024, 512 tiles 36 / 33, 1024 46 / 47,
    // 4096 105 / 118; 75 x 128 x 512 x 512 799 / 990 (4 waves 845).  The line that
    // suits an image moves up with the receivers that a wave walks and with its
    // shape; this one, for all, is within 16 % of the better side.
    int nw = ntiles * passes > 1024 ? 8 : 16;
    w.group = 1;
    while (w.group < 32 && ntiles >= 64 * (int64_t)w.group) w.group *= 2;
    if (sum == WS_BOTH && a.ntx < 8) {
        // few transmits: the receivers are the inner axis and the waves split them
        w.inner_tx = 0;
        w.split_inner = 1;
    } else {
        w.inner_tx = a.sumflag != PYCBF_SUM_RX_ONLY;
    }
    const int ni = w.inner_tx ? a.ntx : a.nrx, no = w.inner_tx ? a.nrx : a.ntx;
    if (!w.split_inner)
        while (nw > 4 && nw / 2 >= no) nw /= 2;
    const int cap = std::min(WAVE_IB, 160 / (w.weights ? 2 : 1));
    const int blocks = (ni + cap - 1) / cap;
    w.ib = blocks == 1 ? ni : ((ni + blocks - 1) / blocks + 15) / 16 * 16;
    // More workgroups than tiles when the tiles alone leave the chip short of
    // waves: the outer axis in chunks, whose sums over both axes go through
    // partial images (as many as the caller's workspace holds).
    const int64_t waves = ntiles * nw * passes;
    const int shares = w.split_inner ? no : (no + nw - 1) / nw;
    int64_t target = 4096;
    if (a.nfr >= 4 && !w.split_inner && a.np <= (int64_t)1 << 24) {
        w.slab = wave_slab(gk, a, sum, no, ni, ntiles, passes) &&
                 (sum != WS_BOTH || (partial && max_part >= 8));
        // sums over frames wait on longer loads: 31 x 64 x 1000 onto 4800 pixels, 16
        // frames, nearest per receiver: 4096 / 8192 / 16384 waves 155 / 123 / 107 us
        if (sum != WS_NONE) target = 16384;
    }
    int64_t nchunk = std::min<int64_t>((target + waves - 1) / waves, shares);
    if (sum == WS_BOTH) nchunk = std::min<int64_t>(nchunk, partial ? max_part : 1);
    if (w.slab) nchunk = 8;
    float *final_out = a.out;
    if (sum == WS_BOTH && nchunk > 1) a.out = partial;
    const size_t lds = std::max(wave_lds_bytes(w.ib, w.weights, nw), (size_t)nw * fc * 64 * 4);
    const dim3 grid((unsigned)(w.slab ? ntiles * 8 : ntiles), (unsigned)(w.slab ? 1 : nchunk),
                    (unsigned)passes);
    int rc;
    {
        ProfScope prof("das_gather", s);
        if (gk == GK_CUBIC)
            rc = wave_launch_cubic(a, w, sum, fc, mode, grid, nw, lds, s);
        else if (gk == GK_KORDER || gk == GK_AKIMA)
            rc = wave_launch_hermite(gk, a, w, sum, fc, mode, grid, nw, lds, s);
        else
            rc = wave_launch_sample(gk, a, w, sum, fc, mode, grid, nw, lds, s);
    }
    if (rc || a.out == final_out) return rc;
    return launch_reduce_split(partial, (int)nchunk, (int64_t)a.nfr * a.np, final_out, s);
}

}  // namespace pycbf
