// Delay-multiply-and-sum over the separated (per-rx or per-tx) axis.
// Formulas of examples/advanced_beamforming.ipynb:296-301 (SSR) and
// examples/develope_gpu_slsc_and_dmas_kernels.ipynb:292-303 (power, P-DMAS-SSR);
// lags come from the caller's array (pycbf/gpu/__advanced_engines__.cu:44-56
// used the loop index instead).
//
// k_dmas_cols: a workgroup takes 64 pixels of a frame (one per lane) and holds
// their whole columns im[:, p] in LDS, read once; the SSR's signed square root
// is taken once per element, ssr(a b) = ssr(a) ssr(b), so a pair costs one LDS
// read and one fused multiply-add.  Its waves split the elements in blocks of
// DB (sums over lags) or the lags (one output per lag).  Bound by the issue of
// those two instructions per pair and by the column reads.  96 elements x
// 60 000 pixels x 10 lags: 251 -> 20 us (k_dmas before: two reads through
// L1, a product and a square root per pair).
//
// k_dmas, a lane per pixel, takes the columns that do not fit LDS and short ones
// of many pixels (dmas_short).
#include <math.h>

#include "common.h"

namespace pycbf {

__device__ __forceinline__ float ssr(float q)
{
    const float r = sqrtf(fabsf(q));
    return q > 0.0f ? r : (q < 0.0f ? -r : 0.0f);
}

// one lane per (frame, pixel), columns of any height
__global__ __launch_bounds__(256) void k_dmas(const float *__restrict__ im, int64_t nfr,
                                              int64_t nsep, int64_t np,
                                              const int32_t *__restrict__ lags, int nlag,
                                              int dmastype, int sumlags, float *__restrict__ out)
{
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nfr * np) return;
    const int64_t f = g / np, p = g - f * np;
    const float *col = im + f * nsep * np + p;
    float total = 0.0f;
    for (int l = 0; l < nlag; ++l) {
        const int m = lags[l];
        float s = 0.0f;
        if (m > 0 && (int64_t)m < nsep) {
            for (int64_t i = 0; i + m < nsep; ++i) {
                const float q = col[i * np] * col[(i + m) * np];
                s += (dmastype == PYCBF_DMAS_SSR) ? ssr(q) : q;
            }
        }
        if (sumlags)
            total += s;
        else
            out[(f * nlag + l) * np + p] = (dmastype == PYCBF_DMAS_PSSR) ? ssr(s) : s;
    }
    if (sumlags) out[f * np + p] = (dmastype == PYCBF_DMAS_PSSR) ? ssr(total) : total;
}

constexpr int DW = 4;          // waves per workgroup
constexpr int DB = 8;          // elements a wave holds in registers
constexpr int DMAX_SEP = 256;  // columns of 64 pixels within 64 KB of LDS

// One product of the pair sum.  GUARD: a signed root of an infinite element
// times one of zero (or of NaN, whose root counts as zero) is NaN where the
// root of their product is zero.
template <bool GUARD>
__device__ __forceinline__ float pair_add(float a, float b, float s)
{
    if (!GUARD) return __builtin_fmaf(a, b, s);
    const float q = a * b;
    return (q == q) ? s + q : s;
}

// sum over the elements i0 .. i0 + DB - 1 of the products at lag m (summed
// apart and added whole: short chains keep the rounding below that of one
// running sum per lag)
template <bool GUARD>
__device__ __forceinline__ float block_sum(const float (&a)[DB], const float *col, int i0, int m,
                                           int nsep)
{
    float s = 0.0f;
    if (i0 + DB - 1 + m < nsep) {
#pragma unroll
        for (int j = 0; j < DB; ++j) s = pair_add<GUARD>(a[j], col[(i0 + j + m) * 64], s);
    } else {
#pragma unroll
        for (int j = 0; j < DB; ++j)
            if (i0 + j + m < nsep) s = pair_add<GUARD>(a[j], col[(i0 + j + m) * 64], s);
    }
    return s;
}

template <bool GUARD>
__device__ __forceinline__ void dmas_sums(const float *col, int nsep, const int32_t *lags,
                                          int nlag, int dmastype, int sumlags, int wave, bool act,
                                          float *red, float *out, int64_t np)
{
    auto fetch = [&](int i0, float(&a)[DB]) {
#pragma unroll
        for (int j = 0; j < DB; ++j) a[j] = col[min(i0 + j, nsep - 1) * 64];
    };
    if (sumlags) {
        float s = 0.0f;
        for (int i0 = wave * DB; i0 < nsep; i0 += DW * DB) {
            float a[DB];
            fetch(i0, a);
            for (int l = 0; l < nlag; ++l) {
                const int m = lags[l];
                if (m > 0 && m < nsep) s += block_sum<GUARD>(a, col, i0, m, nsep);
            }
        }
        red[0] = s;
        return;
    }
    for (int l = wave; l < nlag; l += DW) {
        const int m = lags[l];
        float s = 0.0f;
        if (m > 0 && m < nsep) {
            for (int i0 = 0; i0 + m < nsep; i0 += DB) {
                float a[DB];
                fetch(i0, a);
                s += block_sum<GUARD>(a, col, i0, m, nsep);
            }
        }
        if (act) out[l * np] = (dmastype == PYCBF_DMAS_PSSR) ? ssr(s) : s;
    }
}

__global__ __launch_bounds__(64 * DW) void k_dmas_cols(const float *__restrict__ im, int nsep,
                                                       int64_t np,
                                                       const int32_t *__restrict__ lags, int nlag,
                                                       int dmastype, int sumlags,
                                                       float *__restrict__ out)
{
    extern __shared__ float cols[];  // (nsep, 64), then (DW, 64) wave sums
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t f = blockIdx.y, p = (int64_t)blockIdx.x * 64 + lane;
    const bool act = p < np;
    const float *src = im + f * nsep * np + (act ? p : 0);
    bool inf = false;
#pragma unroll 8
    for (int i = wave; i < nsep; i += DW) {
        float v = act ? src[(int64_t)i * np] : 0.0f;
        if (dmastype == PYCBF_DMAS_SSR) {
            inf = inf || fabsf(v) == INFINITY;
            v = ssr(v);
        }
        cols[i * 64 + lane] = v;
    }
    const bool guard = __syncthreads_or(inf) != 0;
    const float *col = cols + lane;
    float *red = cols + (nsep + wave) * 64 + lane;
    float *o = out + (sumlags ? f : f * nlag) * np + p;
    if (guard)
        dmas_sums<true>(col, nsep, lags, nlag, dmastype, sumlags, wave, act, red, o, np);
    else
        dmas_sums<false>(col, nsep, lags, nlag, dmastype, sumlags, wave, act, red, o, np);
    if (!sumlags) return;  // workgroup-uniform
    __syncthreads();
    if (wave == 0 && act) {
        float s = red[0];
        for (int v = 1; v < DW; ++v) s += red[v * 64];
        *o = (dmastype == PYCBF_DMAS_PSSR) ? ssr(s) : s;
    }
}

// Columns so short that holding them costs more than it saves: k_dmas_cols
// launches four waves per 64 pixels, which many pixels pay for (times over those
// of k_dmas, signed roots, lags 1 .. nsep - 1, summed / apart; n pixels in all):
//   nsep 2: 1.2 at 1000, 3.1 at 1.6 M;  nsep 3: 1.08 / 0.97 at 4000, 1.3 at 100 000
//   nsep 5: 0.9 / 0.7 at 20 000, 1.5 / 1.25 at 400 000, 1.9 / 1.6 at 1.6 M
//   nsep 7: 0.9 / 0.8 at 100 000, 1.2 / 1.0 at 400 000, 1.4 / 1.1 at 1.6 M
//   nsep 9: 0.8 / 0.6 at 100 000, 1.04 / 0.8 at 400 000;  nsep 12: 0.8 / 0.6 at 1.6 M
static bool dmas_short(int64_t nsep, int64_t n, int sumlags)
{
    return nsep < 3 || (nsep <= (sumlags ? 9 : 6) && n >= 32768 * (nsep - 2));
}

int launch_dmas(const float *im, int64_t nfr, int64_t nsep, int64_t np, const int32_t *lags,
                int nlag, int dmastype, int sumlags, float *out, hipStream_t s)
{
    const int64_t n = nfr * np;
    if (n <= 0) return 0;
    // columns too tall for LDS or too short for it, or more frames than a grid axis:
    // through L1
    if (nsep <= DMAX_SEP - DW && nfr <= 65535 && np <= (int64_t)1 << 30 &&
        !dmas_short(nsep, n, sumlags)) {
        const dim3 grid((unsigned)((np + 63) / 64), (unsigned)nfr);
        hipLaunchKernelGGL(k_dmas_cols, grid, dim3(64 * DW), (size_t)(nsep + DW) * 256, s, im,
                           (int)nsep, np, lags, nlag, dmastype, sumlags, out);
        return check_launch("dmas");
    }
    hipLaunchKernelGGL(k_dmas, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, im, nfr, nsep,
                       np, lags, nlag, dmastype, sumlags, out);
    return check_launch("dmas");
}

}  // namespace pycbf
