// Delay and apodisation gradients of the DAS adjoint (das_bwd.hip) on wave
// tiles: one wave per 64 pixels of an outer element, the inner axis' delays and
// weights once per tile in LDS (das_wave.h describes the scheme).  Gradients
// are the sums
//   d tau_o[p] = sum_i,f G w v'(x)      d apod_o[p] = sum_i,f G apod_i v(x)
// over the inner elements in ascending order, frames innermost, in one float32
// chain per (outer element, pixel): the order in which the tables' and the
// geometry's gradients agree bit for bit.  With the geometry, the launches also
// give d loss / d c0 (see k_das_bwd_tau).
//
// The kernel before it (one lane per outer element and pixel, the inner axis
// read or evaluated again for every pair) took 110 - 145 us a launch on 16 x 64 x
// 2048 onto 192 x 256, linear, geometry in registers: 67 us.  Bound as
// the wave-tile gather is: VALU per contributing sample, and L1 lookups.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "das_wave.h"

namespace pycbf {

struct ElemArgs {
    int outer_tx;     // gradients of the transmit elements (else the receive ones)
    int ib;           // inner elements per LDS block
    int weights;      // inner weights in LDS (else they are 1 where a delay is kept)
    uint32_t group;   // neighbouring tiles dealt to one XCD together
    float nhalf;      // nt - 1/2 (nearest)
    const int *fast;  // length of the pixels' fast axis (device), or null
};

// value (v) and derivative (d) of the interpolant; the operations of interp_vd
template <int GK, int MODE>
__device__ __forceinline__ void elem_vd(const BwdArgs &A, const WavePos &P, const WaveRaw &r,
                                        float &v, float &d)
{
    auto over_dt = [&](float u) { return MODE == WM_DIV ? u / A.dt : div_rn(u, A.dt, A.rdt); };
    v = wave_value<GK, GK == GK_LINEAR>(P, r);
    if (GK == GK_NEAREST) {
        d = 0.0f;
    } else if (GK == GK_KORDER || GK == GK_AKIMA) {
        d = __builtin_fmaf(__builtin_fmaf(3.0f * r.v[3], P.a, 2.0f * r.v[2]), P.a, r.v[1]) * A.rdt;
    } else if (GK == GK_LINEAR) {
        const float y0 = P.edge ? r.v[1] : r.v[0], y1 = P.edge ? 0.0f : r.v[1];
        d = over_dt(y1 - y0);
    } else {
        const float da = __builtin_fmaf(3.0f * P.a, P.a, -1.0f);
        const float db = __builtin_fmaf(3.0f * P.b, P.b, -1.0f);
        d = ((r.v[2] - r.v[0]) + (db * r.v[3] - da * r.v[1])) * A.rdt;
    }
}

// Derivative at the position q held in double (delay residuals), as interp_d_at:
// the piece floor(q) with the exact weights
template <int GK>
__device__ __forceinline__ WavePos fine_pos(const BwdArgs &A, double q)
{
    WavePos P;
    P.in = true;
    const int j = min(max((int)floor(q), 0), A.nt - 1);
    const double fr = q - (double)j;
    P.b = (float)fr;
    P.a = (GK == GK_KORDER || GK == GK_AKIMA) ? (float)fr : (float)(1.0 - fr);
    P.c = P.d = 0.0f;
    P.edge = GK == GK_LINEAR && j > A.nt - 2;
    P.off = (uint32_t)(GK == GK_LINEAR ? min(j, A.nt - 2) : j);
    return P;
}

template <int GK>
__device__ __forceinline__ float fine_d(const BwdArgs &A, const WavePos &P, const WaveRaw &r)
{
    if (GK == GK_LINEAR) {
        const float y0 = P.edge ? r.v[1] : r.v[0], y1 = P.edge ? 0.0f : r.v[1];
        return (y1 - y0) * A.rdt;
    }
    float v, d;
    elem_vd<GK, WM_RECIP>(A, P, r, v, d);
    return d;
}

// FINE: delay residuals (tables only)
template <int GK, bool GEOM, int MODE, bool FINE>
__global__ __launch_bounds__(1024) void k_bwd_elem(BwdArgs A, ElemArgs E)
{
    extern __shared__ float sm[];
    constexpr int U = FINE ? 2 : 4;  // inner elements in flight (one frame)
    constexpr int GEO = GEOM ? 3 : 0;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nw = blockDim.x >> 6;
    uint32_t tile = blockIdx.x;
    {
        const uint32_t g = E.group, s8 = tile >> 3;
        if (tile < gridDim.x / (8u * g) * (8u * g))
            tile = ((s8 / g) * 8u + (tile & 7u)) * g + s8 % g;
    }
    const int64_t np = A.np, pos = (int64_t)tile * 64 + lane;
    const bool act = pos < np;
    int64_t p = 0;
    if (act) {
        const int fast = E.fast ? *E.fast : 0;
        p = fast ? band_pixel(pos, np, fast) : pos;
    }
    float pv[3] = {0.0f, 0.0f, 0.0f};
    if (GEOM) {
        for (int d = 0; d < A.geo; ++d) {
            const float v = A.pvec[p * A.geo + d];
            if (d == 0) pv[0] = v;
            else if (d == 1) pv[1] = v;
            else pv[2] = v;
        }
    }
    DasArgs D{};  // the forward's view of the same arrays and axes
    D.ttx = A.ttx;
    D.atx = A.atx;
    D.trx = A.trx;
    D.arx = A.arx;
    D.np = np;
    D.txpack = A.txpack;
    D.rxpack = A.rxpack;
    D.c0 = A.c0;
    D.t0 = A.t0;
    D.dt = A.dt;
    D.rdt = A.rdt;
    D.tmax = A.tmax;
    D.nsrc = A.nt;
    const bool otx = E.outer_tx != 0;
    const int no = otx ? A.ntx : A.nrx, ni = otx ? A.nrx : A.ntx;
    const bool drop = A.thresh > 0.0f;  // a zero (or NaN) weight then never contributes
    float *s_tau = sm;
    float *s_ap = sm + E.ib * 64;
    float *s_lo = s_ap + (E.weights ? E.ib * 64 : 0);
    int *s_any = reinterpret_cast<int *>(s_lo + (FINE ? E.ib * 64 : 0));
    constexpr int BYTES = GK == GK_CUBIC ? 8 : (GK == GK_KORDER || GK == GK_AKIMA ? 16 : 4);
    const int64_t rowb = (int64_t)(GK == GK_CUBIC ? A.nt + 1 : A.nt) * BYTES;
    const int64_t ibytes = (otx ? 1 : (int64_t)A.nrx) * rowb;
    const int64_t obytes = (otx ? (int64_t)A.nrx : 1) * rowb;
    const int64_t fbytes = (int64_t)A.ntx * A.nrx * rowb;
    // upstream gradient: element (i, f) of this outer element at gi * i + gf * f + base
    const bool g_in = A.sumflag == PYCBF_SUM_NONE ||
                      A.sumflag == (otx ? PYCBF_SUM_TX_ONLY : PYCBF_SUM_RX_ONLY);
    const double rdt_d = 1.0 / (double)A.dt;
    const float *lo_o = otx ? A.ttx_lo : A.trx_lo, *lo_i = otx ? A.trx_lo : A.ttx_lo;
    double c0sum = 0.0;

    for (int i0 = 0; i0 < ni; i0 += E.ib) {
        const int n = min(E.ib, ni - i0);
        const bool last = i0 + E.ib >= ni;
        if (i0) __syncthreads();
        for (int k = wave; k < n; k += nw) {
            float tau, ap;
            elem_eval<GEO>(D, !otx, i0 + k, p, pv, tau, ap);
            if (!act || (drop && !(ap != 0.0f && ap == ap))) tau = NAN;
            s_tau[k * 64 + lane] = tau;
            if (E.weights) s_ap[k * 64 + lane] = ap;
            if (FINE) s_lo[k * 64 + lane] = lo_i ? lo_i[(int64_t)(i0 + k) * np + p] : 0.0f;
            const int any = __any(tau == tau) ? 1 : 0;
            if (lane == 0) s_any[k] = any;
        }
        __syncthreads();
        for (int o = (int)blockIdx.y + (int)gridDim.y * wave; o < no; o += (int)gridDim.y * nw) {
            float to, wo;
            elem_eval<GEO>(D, otx, o, p, pv, to, wo);
            const float tau_o = to;
            if (!act || (drop && !(wo != 0.0f && wo == wo))) to = NAN;
            const double lod = (FINE && lo_o) ? (double)lo_o[(int64_t)o * np + p] : 0.0;
            float gt = 0.0f, ga = 0.0f;
            if (i0 && act) {  // the chain goes on from the blocks before
                if (A.gtau) gt = A.gtau[(int64_t)o * np + p];
                if (A.gapod) ga = A.gapod[(int64_t)o * np + p];
            }
            const int64_t gbase = A.sumflag == PYCBF_SUM_NONE
                                      ? (otx ? (int64_t)o * A.nrx : (int64_t)o) * np
                                      : (g_in || A.sumflag == PYCBF_SUM_TX_AND_RX ? 0 : o * np);
            const int64_t gi = !g_in ? 0
                               : (A.sumflag == PYCBF_SUM_NONE && !otx ? (int64_t)A.nrx * np : np);
            const int64_t gf = A.sumflag == PYCBF_SUM_NONE ? (int64_t)A.ntx * A.nrx * np
                               : A.sumflag == PYCBF_SUM_TX_AND_RX ? np
                               : A.sumflag == PYCBF_SUM_TX_ONLY   ? (int64_t)A.nrx * np
                                                                  : (int64_t)A.ntx * np;
            const float *gp = A.gout + gbase + p;
            const char *row0 = reinterpret_cast<const char *>(A.src) + (int64_t)i0 * ibytes +
                               (int64_t)o * obytes;
            float g0 = (!g_in && A.nfr == 1) ? gp[0] : 0.0f;
            auto group = [&](const int *k, auto nuc) {
                constexpr int NU = decltype(nuc)::value;
                WavePos P[NU], Q[NU];
                float w[NU], ap[NU];
#pragma unroll
                for (int u = 0; u < NU; ++u) {
                    const float ti = s_tau[k[u] * 64 + lane];
                    ap[u] = E.weights ? s_ap[k[u] * 64 + lane] : 1.0f;
                    w[u] = ap[u] * wo;
                    const float x = ti + to;
                    P[u] = wave_pos<GK, MODE, GK == GK_LINEAR, false>(D, E.nhalf, x);
                    P[u].in = P[u].in && fabsf(w[u]) >= A.thresh;
                    if (FINE) {
                        const double xd = ((double)ti + (double)to) +
                                          (lod + (double)s_lo[k[u] * 64 + lane]);
                        Q[u] = fine_pos<GK>(A, P[u].in ? (xd - (double)A.t0) * rdt_d : 0.0);
                    }
                }
                for (int f = 0; f < A.nfr; ++f) {
                    WaveRaw R[NU], F[NU];
                    float g[NU];
#pragma unroll
                    for (int u = 0; u < NU; ++u) {
                        const char *row = row0 + f * fbytes + (int64_t)k[u] * ibytes;
                        if (!FINE || A.gapod)
                            R[u] = wave_load<GK, MODE>(row - WAVE_OFF_BITS, P[u].off);
                        if (FINE) F[u] = wave_load<GK, WM_DIV>(row - WAVE_OFF_BITS, Q[u].off);
                        g[u] = (!g_in && A.nfr == 1) ? g0 : gp[(i0 + k[u]) * gi + f * gf];
                    }
#pragma unroll
                    for (int u = 0; u < NU; ++u) {
                        float v = 0.0f, d = 0.0f;
                        if (!FINE || A.gapod) elem_vd<GK, MODE>(A, P[u], R[u], v, d);
                        if (FINE) d = fine_d<GK>(A, Q[u], F[u]);
                        const float t = __builtin_fmaf(g[u] * w[u], d, gt);
                        const float a = __builtin_fmaf(g[u] * ap[u], v, ga);
                        gt = P[u].in ? t : gt;
                        ga = P[u].in ? a : ga;
                    }
                }
            };
            if (__any(to == to)) {
#pragma unroll 1
                for (int w = 0; w < n; w += 64) {
                    // the elements some lane of the tile uses
                    const uint64_t b = __ballot(w + lane < n && s_any[w + lane]);
                    uint64_t m = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32) |
                                 (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b);
                    int left = __popcll(m);
                    int k[U];
                    for (; A.nfr == 1 && left >= U; left -= U) {
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            k[u] = w + __builtin_ctzll(m);
                            m &= m - 1;
                        }
                        group(k, std::integral_constant<int, U>());
                    }
                    for (; left > 0; --left) {
                        k[0] = w + __builtin_ctzll(m);
                        m &= m - 1;
                        group(k, std::integral_constant<int, 1>());
                    }
                }
            }
            if (act && A.gtau) A.gtau[(int64_t)o * np + p] = gt;
            if (act && A.gapod) A.gapod[(int64_t)o * np + p] = ga;
            if (GEOM && last && A.gc0part && act && gt != 0.0f)
                c0sum += (double)gt * (-(double)tau_o / (double)A.c0);
        }
    }
    if (GEOM && A.gc0part) {
        // fixed-order workgroup sum in double: wave butterflies, then the waves
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) c0sum += __shfl_xor(c0sum, off, 64);
        __shared__ double wsum[16];
        if (lane == 0) wsum[wave] = c0sum;
        __syncthreads();
        if (threadIdx.x == 0) {
            double c = wsum[0];
            for (int v = 1; v < nw; ++v) c += wsum[v];
            A.gc0part[A.gc0_off + (int64_t)blockIdx.y * gridDim.x + blockIdx.x] = c;
        }
    }
}

template <int GK, bool GEOM, bool FINE>
static void elem_mode(int mode, const BwdArgs &a, const ElemArgs &e, dim3 grid, dim3 block,
                      size_t lds, hipStream_t s)
{
    if (mode == WM_RECIP0)
        hipLaunchKernelGGL((k_bwd_elem<GK, GEOM, WM_RECIP0, FINE>), grid, block, lds, s, a, e);
    else if (mode == WM_RECIP)
        hipLaunchKernelGGL((k_bwd_elem<GK, GEOM, WM_RECIP, FINE>), grid, block, lds, s, a, e);
    else
        hipLaunchKernelGGL((k_bwd_elem<GK, GEOM, WM_DIV, FINE>), grid, block, lds, s, a, e);
}

template <int GK>
static void elem_geo(bool fine, int mode, const BwdArgs &a, const ElemArgs &e, dim3 grid,
                     dim3 block, size_t lds, hipStream_t s)
{
    if (a.geo)
        elem_mode<GK, true, false>(mode, a, e, grid, block, lds, s);
    else if (fine)
        elem_mode<GK, false, true>(mode, a, e, grid, block, lds, s);
    else
        elem_mode<GK, false, false>(mode, a, e, grid, block, lds, s);
}

int launch_bwd_elem(int gk, const BwdArgs &a, int outer_tx, int &parts, hipStream_t s)
{
    parts = 0;
    if (gk == GK_LINEAR && a.nt < 2) return 1;          // reads pairs
    if (gk == GK_NEAREST && a.nt > 1 << 22) return 1;   // nt - 1/2 as a float
    if (a.np > (int64_t)1 << 28) return 1;
    const bool fine = a.geo == 0 && (a.ttx_lo || a.trx_lo) && gk != GK_NEAREST;
    const int ni = outer_tx ? a.nrx : a.ntx, no = outer_tx ? a.ntx : a.nrx;
    ElemArgs e{};
    e.outer_tx = outer_tx;
    e.weights = !(a.geo && a.thresh > 0.0f && a.thresh <= 1.0f);
    e.nhalf = (float)a.nt - 0.5f;
    // LDS rows: 48 KB per workgroup.  Blocks go on from the gradients stored by
    // the one before; without a delay gradient to store (c0 alone) one block has
    // to hold the axis.
    const int row = 256 * (1 + (e.weights ? 1 : 0) + (fine ? 1 : 0)) + 4;
    const bool one = a.gc0part && !a.gtau;
    const int cap = (one ? 150 * 1024 : 48 * 1024) / row;
    if (one && ni > cap) return 1;
    const int blocks = (ni + cap - 1) / cap;
    e.ib = (ni + blocks - 1) / blocks;
    const int64_t ntiles = (a.np + 63) / 64;
    e.group = 1;
    while (e.group < 32 && ntiles >= 64 * (int64_t)e.group) e.group *= 2;
    int nw = ntiles > 1024 ? 8 : 16;
    while (nw > 4 && nw / 2 >= no) nw /= 2;
    const int64_t waves = ntiles * nw;
    const int64_t nchunk = std::min<int64_t>({(4096 + waves - 1) / waves, (no + nw - 1) / nw, 8});
    e.fast = a.fast;
    parts = (int)(ntiles * nchunk);
    const int mode = wave_mode_of(a.t0, a.dt, a.rdt, a.tmax, a.nt);
    const dim3 grid((unsigned)ntiles, (unsigned)nchunk), block((unsigned)nw * 64);
    const size_t lds = (size_t)e.ib * row;
    switch (gk) {
    case GK_NEAREST: elem_geo<GK_NEAREST>(fine, mode, a, e, grid, block, lds, s); break;
    case GK_LINEAR: elem_geo<GK_LINEAR>(fine, mode, a, e, grid, block, lds, s); break;
    case GK_KORDER: elem_geo<GK_KORDER>(fine, mode, a, e, grid, block, lds, s); break;
    case GK_AKIMA: elem_geo<GK_AKIMA>(fine, mode, a, e, grid, block, lds, s); break;
    default: elem_geo<GK_CUBIC>(fine, mode, a, e, grid, block, lds, s); break;
    }
    return check_launch("das_bwd_elem");
}

}  // namespace pycbf
