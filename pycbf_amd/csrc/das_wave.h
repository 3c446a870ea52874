// Wave-tile gather: one wave owns 64 pixels (a compact 8 x 8 patch in the
// processing order), one per lane, and reads each sample straight from the
// channel's row through L1.
//
// A workgroup of nw waves shares one pixel tile.  The delays (and weights) of
// one channel axis, the inner one, are evaluated once per tile into LDS, one
// float per (element, lane), so a channel costs one conflict-free LDS read
// instead of a table read or a geometry evaluation; the waves walk the other,
// outer axis with that element's delay in a register.  An element that no
// lane of the tile can use is dropped before the channel loop: the inner ones
// from a bit mask (scalar bit scans, so a channel's row address is scalar
// arithmetic), the outer ones by a wave-uniform test.  A lane that does not
// use an element holds a NaN delay: it fails the trace test, so a sample
// needs no weight test of its own (and where the tile's delay range shows that
// every sample of the wave lies on the trace, no trace test either).  Delays
// are clamped to the trace and results selected, so the loads of the unrolled
// channels and of all frames are in flight together.
//
// What bounds it: per wave and contributing channel about 23 VALU
// instructions (cubic; 13 k-order) and the L1 lookups of a 64-lane gather of
// 16-byte entries (22 lines measured, 16 at best), and the L2 latency of
// about three lines per gather that the waves in flight must cover.
// One frame of 75 x 128 x 4096 onto 512 x 512, cubic: 1.84 -> 0.70 ms (the
// gather with transmit delays in registers before it: 0.48 T wave-level VALU
// instructions at 30 per sample, and no dropped elements); 31 x 128 x 2048 onto
// 256 x 256, k-order: 700 -> 117 us (staged through LDS, one barrier per
// channel, before); 15 x 96 x 2048, linear per-receive images: 248 -> 75 us.
//
// The frames' sums stay in registers.  tx_and_rx adds the waves' sums in LDS
// in a fixed order and stores the image once, with no clear and no atomics.
//
// Sample selection, knot times and weights are the float32 operations of
// pycbf/cpu/pycbf.c:68-105,179-271 (see gather() in das_dev.h).
#pragma once
#include <math.h>

#include "common.h"
#include "das_dev.h"
#include "prof.h"

namespace pycbf {

struct WaveArgs {
    int inner_tx;     // transmits are the inner (LDS) axis
    int split_inner;  // the waves split the inner elements, not the outer ones
    int ib;           // inner elements per LDS block (<= WAVE_IB)
    uint32_t group;   // neighbouring tiles dealt to one XCD together
    int slab;         // 8 chunks of the outer axis, one per XCD
    int weights;      // inner weights are stored in LDS (tables, or thresh outside (0, 1])
    float nhalf;      // nsrc - 1/2 (nearest)
    const int *fast;  // length of the pixels' fast axis (device, 0: unknown), or null
};

// Pixel of position i of the order that cuts a grid of np / fast lines of
// `fast` pixels into bands of 8 lines, along the fast axis first: 64 positions
// are an 8 x 8 patch (the last band may hold fewer lines).
__device__ __forceinline__ int64_t band_pixel(int64_t i, int64_t np, int fast)
{
    const int64_t band = i / (8 * (int64_t)fast), r = i - band * 8 * fast;
    const int64_t left = np / fast - 8 * band;
    const uint32_t w = left < 8 ? (uint32_t)left : 8u;
    const uint32_t z = (uint32_t)r / w, c = (uint32_t)r - z * w;
    return (band * 8 + c) * fast + z;
}

// channels whose samples a wave has in flight (one frame).  The gather waits on
// L1 and L2 latency more than it computes: 4 / 5 / 6 / 8 channels take 799 /
// 802 / 815 / 882 us on 75 x 128 x 512 x 512 (cubic) and 218 / 208 / 208 / 262 us
// on 31 x 128 x 128 x 1024 per-receive images; 8 costs occupancy.
constexpr int WAVE_U = 5;
constexpr int WAVE_IB = 192;  // three 64-bit masks
// A row offset is formed in float: fma(index, bytes, 2^23) holds it in its low
// bits, in one instruction and with no conversion to integer; the row pointers
// are lowered by the bits of 2^23.  Byte offsets (16 per entry) below 2^23:
// traces of up to 2^19 entries; longer ones take WM_DIV.
constexpr int64_t WAVE_FLOAT_NSRC = (int64_t)1 << 19;
constexpr float WAVE_OFF_BIAS = 8388608.0f;
constexpr uint32_t WAVE_OFF_BITS = 0x4b000000u;

// output classes: summed over both axes, one image per outer element, every
// (tx, rx) pair
enum WaveSum { WS_BOTH = 0, WS_SEP = 1, WS_NONE = 2 };

// quotients by dt: the division (with the knot index clamped to the trace, and
// integer offsets: every trace), products with the reciprocal (dt accepted by
// recip_division_exact: the same quotients; wave_mode_of says when), and those
// with t0 = 0
enum WaveMode { WM_DIV = 0, WM_RECIP = 1, WM_RECIP0 = 2 };

// The mode for a trace of nsrc entries; host only.  The reciprocal modes do not
// clamp the knot index, so the last sample time itself must select a knot (a
// quotient that is no number does not).
inline int wave_mode_of(float t0, float dt, float rdt, float tmax, int64_t nsrc)
{
    if (nsrc > WAVE_FLOAT_NSRC || !((tmax - t0) / dt < (float)nsrc)) return WM_DIV;
    if (rdt != 1.0f / dt || !recip_division_exact(dt)) return WM_DIV;
    return t0 == 0.0f ? WM_RECIP0 : WM_RECIP;
}

// a sample's place in its row and what its value needs
struct WavePos {
    uint32_t off;         // bytes into the row plus WAVE_OFF_BITS (WM_DIV: the entry)
    float a, b, c, d;     // interpolation weights (or the Hermite position)
    bool in, edge;
};

// entry j (jf as a float) of a row with entries of `bytes`
template <int MODE>
__device__ __forceinline__ uint32_t wave_off(int j, float jf, float bytes)
{
    if (MODE == WM_DIV) return (uint32_t)j;
    return __float_as_uint(__builtin_fmaf(jf, bytes, WAVE_OFF_BIAS));
}

// INSIDE: every lane's x is known to lie on the trace, and for nearest also to
// round to one of its entries (a last sample time that float rounding has moved
// up by half a sample or more rounds to the entry after them)
template <int GK, int MODE, bool EXACT, bool INSIDE>
__device__ __forceinline__ WavePos wave_pos(const DasArgs &A, float nhalf, float x)
{
    WavePos P;
    P.edge = false;
    P.in = true;
    P.a = P.b = P.c = P.d = 0.0f;
    const float t0 = MODE == WM_RECIP0 ? 0.0f : A.t0;
    auto over_dt = [&](float v) { return MODE == WM_DIV ? v / A.dt : div_rn(v, A.dt, A.rdt); };
    if (GK == GK_NEAREST) {
        // (int)(q + 0.5) with the 0.5 added in double, for -1 < q + 0.5 < nsrc:
        // trunc(q) plus one when the exact fraction reaches 1/2, and 0 below 0
        const float q = over_dt(MODE == WM_RECIP0 ? x : x - t0);
        float qc = q;
        if (!INSIDE) {
            P.in = q > -1.5f && q < nhalf;
            qc = __builtin_amdgcn_fmed3f(q, 0.0f, nhalf - 0.5f);
        }
        const float jf = truncf(qc);
        const float it = (qc - jf >= 0.5f) ? jf + 1.0f : jf;
        P.off = wave_off<MODE>((int)it, it, 4.0f);
        return P;
    }
    float xc = x;
    if (!INSIDE) {
        xc = __builtin_amdgcn_fmed3f(x, t0, A.tmax);
        P.in = xc == x;
    }
    const float q = over_dt(MODE == WM_RECIP0 ? xc : xc - t0);
    const int j = MODE == WM_DIV ? min((int)q, A.nsrc - 1) : 0;
    const float jf = MODE == WM_DIV ? (float)j : truncf(q);
    if (GK == GK_KORDER || GK == GK_AKIMA) {
        if (MODE == WM_RECIP0)
            P.a = (xc - A.dt * jf) * A.rdt;
        else
            P.a = (GK == GK_KORDER) ? ((xc - t0) - A.dt * jf) * A.rdt
                                    : (xc - (t0 + A.dt * jf)) * A.rdt;
        P.off = wave_off<MODE>(j, jf, 16.0f);
        return P;
    }
    const float lead = A.dt * (jf + 1.0f), lag = A.dt * jf;
    const float xlead = MODE == WM_RECIP0 ? lead : t0 + lead;
    const float xlag = MODE == WM_RECIP0 ? lag : t0 + lag;
    if (GK == GK_LINEAR) {
        P.a = EXACT ? over_dt(xlead - xc) : (xlead - xc) * A.rdt;
        P.b = EXACT ? over_dt(xc - xlag) : (xc - xlag) * A.rdt;
        // the pair (nsrc - 2, nsrc - 1) serves the last knot, whose successor is 0
        const float last = nhalf - 1.5f;
        P.edge = MODE == WM_DIV ? j > A.nsrc - 2 : jf > last;
        P.off = wave_off<MODE>(min(j, A.nsrc - 2), fminf(jf, last), 4.0f);
        return P;
    }
    P.a = (xlead - xc) * A.rdt;
    P.b = (xc - xlag) * A.rdt;
    P.c = __builtin_fmaf(P.a * P.a, P.a, -P.a);
    P.d = __builtin_fmaf(P.b * P.b, P.b, -P.b);
    P.off = wave_off<MODE>(j, jf, 8.0f);
    return P;
}

typedef __attribute__((address_space(3))) float lds_float;

struct WaveRaw {
    float v[4];
};
// a row's entries as read: pairs at 4-byte, (y, h*y2) pairs at 8-byte alignment
typedef float wave_f2 __attribute__((ext_vector_type(2), aligned(4)));
typedef float wave_f4a8 __attribute__((ext_vector_type(4), aligned(8)));
typedef float wave_f4 __attribute__((ext_vector_type(4), aligned(16)));

template <int GK, int MODE>
__device__ __forceinline__ WaveRaw wave_load(const char *row, uint32_t o)
{
    constexpr int BYTES = GK == GK_CUBIC ? 8 : (GK == GK_KORDER || GK == GK_AKIMA ? 16 : 4);
    // rows are global memory, also where the compiler cannot see it
#define WAVE_AT(T) (*(const __attribute__((address_space(1))) T *)((uintptr_t)row + off))
    const size_t off = MODE == WM_DIV ? (size_t)o * BYTES + WAVE_OFF_BITS : (size_t)o;
    WaveRaw r;
    if (GK == GK_NEAREST) {
        r.v[0] = WAVE_AT(float);
    } else if (GK == GK_LINEAR) {
        const wave_f2 p = WAVE_AT(wave_f2);
        r.v[0] = p.x;
        r.v[1] = p.y;
    } else if (GK == GK_CUBIC) {
        const wave_f4a8 p = WAVE_AT(wave_f4a8);  // y_j, z_j, y_j+1, z_j+1
        r.v[0] = p.x;
        r.v[1] = p.y;
        r.v[2] = p.z;
        r.v[3] = p.w;
    } else {
        const wave_f4 p = WAVE_AT(wave_f4);
        r.v[0] = p.x;
        r.v[1] = p.y;
        r.v[2] = p.z;
        r.v[3] = p.w;
    }
#undef WAVE_AT
    return r;
}

// the sample's value plus s; CHAIN: the cubic's own sum starts from s (one
// instruction less), else the value is added whole
template <int GK, bool EXACT>
__device__ __forceinline__ float wave_value(const WavePos &P, const WaveRaw &r);

template <int GK, bool CHAIN>
__device__ __forceinline__ float wave_add(const WavePos &P, const WaveRaw &r, float s)
{
    if (GK == GK_CUBIC && CHAIN) {
        s = __builtin_fmaf(P.a, r.v[0], s);
        s = __builtin_fmaf(P.b, r.v[2], s);
        s = __builtin_fmaf(P.c, r.v[1], s);
        return __builtin_fmaf(P.d, r.v[3], s);
    }
    return s + wave_value<GK, false>(P, r);
}

template <int GK, bool EXACT>
__device__ __forceinline__ float wave_value(const WavePos &P, const WaveRaw &r)
{
    if (GK == GK_NEAREST) return r.v[0];
    if (GK == GK_LINEAR) {
        const float y0 = P.edge ? r.v[1] : r.v[0];
        const float y1 = P.edge ? 0.0f : r.v[1];
        return EXACT ? P.a * y0 + P.b * y1 : __builtin_fmaf(P.b, y1, P.a * y0);
    }
    if (GK == GK_CUBIC) {
        float v = P.a * r.v[0];
        v = __builtin_fmaf(P.b, r.v[2], v);
        v = __builtin_fmaf(P.c, r.v[1], v);
        return __builtin_fmaf(P.d, r.v[3], v);
    }
    return __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(r.v[3], P.a, r.v[2]), P.a, r.v[1]), P.a,
                          r.v[0]);
}

// This wave's share of a tile's channels: inner elements ibeg .. iend - 1 (held
// in LDS by the whole workgroup, of which it takes those in `pat`), outer ones
// obeg, obeg + ostep, ... below oend.
struct WaveShare {
    int ibeg, iend, obeg, oend, ostep;
    uint64_t pat;
};

__device__ __forceinline__ uint64_t every_nth(int wave, int nw)
{
    uint64_t pat = 1ull << wave;
    for (int s = nw; s < 64; s <<= 1) pat |= pat << s;
    return pat;
}

// LDS of one workgroup: delays (and weights) of ib inner elements, the waves'
// delay ranges, the elements' flags
__host__ __device__ inline size_t wave_lds_bytes(int ib, int weights, int nw)
{
    return (size_t)ib * 64 * 4 * (weights ? 2 : 1) + (size_t)nw * 128 * 4 + (size_t)ib * 4;
}

// Walks the workgroup's tile (this lane's pixel p at pv): sums of both axes go
// to acc, the other classes to A.out.  All waves of the workgroup call it
// together, and LDS is free when they do.
template <int GK, int SUM, int FC, bool GEOM, int MODE>
__device__ __forceinline__ void wave_sweep(const DasArgs &A, const WaveArgs &W, float *sm,
                                           const WaveShare &share, int nw, int wave, int lane,
                                           bool act, int64_t p, const float (&pv)[3], int f0,
                                           int nf, float (&acc)[FC])
{
    constexpr int U = FC == 1 ? WAVE_U : (FC == 2 ? 2 : 1);  // channels in flight together
    constexpr bool EXACT = SUM == WS_NONE;
    // Single-frame images of one element feed the coherence kernels, whose
    // 16-bit operands turn a last-bit change of an image into 1e-5 of theirs:
    // the order of these sums is part of the result (whole values, added in
    // blocks of 16 inner elements, the blocks then added in order).
    constexpr bool B16 = SUM == WS_SEP && GK == GK_CUBIC && FC == 1;
    constexpr int GEO = GEOM ? 3 : 0;
    const bool inner_tx = W.inner_tx != 0;
    const int no = inner_tx ? A.nrx : A.ntx;
    const bool drop = A.thresh > 0.0f;  // a zero (or NaN) weight then never contributes
    // nearest: whether the last sample time rounds to an entry, as then every
    // earlier one does (quotients are monotone in the time)
    const bool last_in =
        GK != GK_NEAREST || wave_pos<GK, MODE, EXACT, false>(A, W.nhalf, A.tmax).in;
    float *s_tau = sm;
    float *s_wgt = sm + W.ib * 64;
    // this lane's column of s_tau as an LDS address the compiler holds in one
    // register (it would add the array's base again for every channel)
    uint32_t l_tau = (uint32_t)(uintptr_t)(lds_float *)(s_tau + lane);
    asm("" : "+v"(l_tau));
    auto tau_of = [&](int k) { return *(lds_float *)(uintptr_t)(l_tau + ((uint32_t)k << 8)); };
    float *s_rng = sm + W.ib * 64 * (W.weights ? 2 : 1);  // (nw, 64) delay ranges (lo, hi)
    int *s_flag = reinterpret_cast<int *>(s_rng + nw * 128);
    const int64_t fbytes = (int64_t)A.ntx * A.nrx * A.ch_stride * 4;
    const int64_t ibytes = (inner_tx ? (int64_t)A.nrx : 1) * A.ch_stride * 4;
    const int64_t obytes = (inner_tx ? 1 : (int64_t)A.nrx) * A.ch_stride * 4;

    for (int i0 = share.ibeg; i0 < share.iend; i0 += W.ib) {
        const int n = min(W.ib, share.iend - i0);
        if (i0 != share.ibeg) __syncthreads();
        float lo = INFINITY, hi = -INFINITY;  // this lane's delays over the kept elements
        for (int k = wave; k < n; k += nw) {
            float tau, ap;
            elem_eval<GEO>(A, inner_tx, i0 + k, p, pv, tau, ap);
            if (!act || (drop && !(ap != 0.0f && ap == ap))) tau = NAN;
            s_tau[k * 64 + lane] = tau;
            if (W.weights) s_wgt[k * 64 + lane] = ap;
            const int any = __any(tau == tau) ? 1 : 0;
            const int ones = __all(!(tau == tau) || ap == 1.0f) ? 2 : 0;
            if (lane == 0) s_flag[k] = any | ones;
            if (any) {
                lo = (tau == tau) ? fminf(lo, tau) : -INFINITY;
                hi = (tau == tau) ? fmaxf(hi, tau) : INFINITY;
            }
        }
        s_rng[wave * 128 + lane] = lo;
        s_rng[wave * 128 + 64 + lane] = hi;
        __syncthreads();
        for (int v = 0; v < nw; ++v) {
            lo = fminf(lo, s_rng[v * 128 + lane]);
            hi = fmaxf(hi, s_rng[v * 128 + 64 + lane]);
        }
        uint64_t mask[WAVE_IB / 64];
        bool unit = true;
#pragma unroll
        for (int w = 0; w < WAVE_IB / 64; ++w) {
            const int fl = (w * 64 + lane < n) ? s_flag[w * 64 + lane] : 2;
            const uint64_t m =
                __ballot((SUM == WS_NONE) ? (w * 64 + lane < n) : (fl & 1) != 0) & share.pat;
            mask[w] = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(m >> 32)) << 32) |
                      (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)m);
            unit = unit && __all((fl & 2) != 0);
        }
        // all inner weights 1 (or their lanes dropped): samples are summed
        // unweighted and the outer weight is applied to the sum
        if (!W.weights) unit = true;

        for (int o = share.obeg; o < share.oend; o += share.ostep) {
            float to, wo;
            elem_eval<GEO>(A, !inner_tx, o, p, pv, to, wo);
            if (!act || (drop && !(wo != 0.0f && wo == wo))) to = NAN;
            if (unit && !(fabsf(wo) >= A.thresh)) to = NAN;
            // an infinite outer weight goes to every sample: times a sum it would
            // be NaN where no sample counts, or where the sum has lost a sign
            const bool whole = unit && (GEOM || SUM == WS_NONE ||
                                        __all(!(to == to) || fabsf(wo) < INFINITY));
            float part[FC];
#pragma unroll
            for (int f = 0; f < FC; ++f) part[f] = 0.0f;
            const char *row0 = reinterpret_cast<const char *>(A.src) + (int64_t)f0 * fbytes +
                               (int64_t)i0 * ibytes + (int64_t)o * obytes;
            float total = 0.0f;  // B16: the sum of the blocks before k's
            int block = 0;
            // nu channels: positions, then every load, then the values
            auto group = [&](const int *k, auto nuc, auto kindc) {
                constexpr int NU = decltype(nuc)::value;
                constexpr bool UNIT = decltype(kindc)::value >= 1;
                constexpr bool INSIDE = decltype(kindc)::value == 2;
                WavePos P[NU];
                WaveRaw R[NU][FC];
                float wgt[NU];
#pragma unroll
                for (int u = 0; u < NU; ++u) {
                    P[u] = wave_pos<GK, MODE, EXACT, INSIDE>(A, W.nhalf, tau_of(k[u]) + to);
                    wgt[u] = 1.0f;
                    if (!UNIT) {
                        wgt[u] = s_wgt[k[u] * 64 + lane] * wo;  // apodtx * apodrx
                        P[u].in = P[u].in && fabsf(wgt[u]) >= A.thresh;
                    }
                }
#pragma unroll
                for (int u = 0; u < NU; ++u) {
                    const char *row = row0 + (int64_t)k[u] * ibytes - WAVE_OFF_BITS;
#pragma unroll
                    for (int f = 0; f < FC; ++f)
                        R[u][f] = wave_load<GK, MODE>(row + (int64_t)min(f, nf - 1) * fbytes, P[u].off);
                }
#pragma unroll
                for (int u = 0; u < NU; ++u) {
                    if (B16 && (k[u] >> 4) != block) {  // wave-uniform
                        block = k[u] >> 4;
                        total += part[0];
                        part[0] = 0.0f;
                    }
#pragma unroll
                    for (int f = 0; f < FC; ++f) {
                        if (SUM == WS_NONE) {
                            const float v = wave_value<GK, EXACT>(P[u], R[u][f]);
                            const int e = i0 + k[u];
                            const int64_t ch = inner_tx ? (int64_t)e * A.nrx + o
                                                        : (int64_t)o * A.nrx + e;
                            const float w = UNIT ? (GEOM ? 1.0f : wo) : wgt[u];
                            if (act && f < nf)
                                A.out[((int64_t)(f0 + f) * A.ntx * A.nrx + ch) * A.np + p] =
                                    P[u].in ? 0.0f + w * v : 0.0f;
                        } else if (INSIDE) {
                            part[f] = wave_add<GK, !B16>(P[u], R[u][f], part[f]);
                        } else if (UNIT) {
                            const float s = wave_add<GK, !B16>(P[u], R[u][f], part[f]);
                            part[f] = P[u].in ? s : part[f];
                        } else {
                            const float v = wave_value<GK, EXACT>(P[u], R[u][f]);
                            const float s = __builtin_fmaf(wgt[u], v, part[f]);
                            part[f] = P[u].in ? s : part[f];
                        }
                    }
                }
            };
            auto sweep = [&](auto kindc) {
#pragma unroll 1
                for (int w = 0; w < WAVE_IB / 64; ++w) {
                    uint64_t m = w == 0 ? mask[0] : (w == 1 ? mask[1] : mask[2]);
                    int left = __popcll(m);
                    int k[U];
                    for (; left >= U; left -= U) {
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            k[u] = w * 64 + __builtin_ctzll(m);
                            m &= m - 1;
                        }
                        group(k, std::integral_constant<int, U>(), kindc);
                    }
                    for (; U > 2 && left >= 2; left -= 2) {
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            k[u] = w * 64 + __builtin_ctzll(m);
                            m &= m - 1;
                        }
                        group(k, std::integral_constant<int, (U > 2 ? 2 : 1)>(), kindc);
                    }
                    for (; left > 0; --left) {
                        k[0] = w * 64 + __builtin_ctzll(m);
                        m &= m - 1;
                        group(k, std::integral_constant<int, 1>(), kindc);
                    }
                }
                if (B16) part[0] = total + part[0];
            };
            if (SUM == WS_NONE || __any(to == to)) {
                // every sample of the wave on the trace: no clamps, no selects
                const bool inside = SUM != WS_NONE && whole && last_in &&
                                    __all(lo + to >= A.t0 && hi + to <= A.tmax);
                if (inside)
                    sweep(std::integral_constant<int, SUM == WS_NONE ? 1 : 2>());
                else if (whole)
                    sweep(std::integral_constant<int, 1>());
                else
                    sweep(std::integral_constant<int, 0>());
            }
            if (SUM == WS_NONE) continue;
            if (!GEOM && whole) {
#pragma unroll
                for (int f = 0; f < FC; ++f) part[f] *= (to == to) ? wo : 0.0f;
            }
            if (SUM == WS_BOTH) {
#pragma unroll
                for (int f = 0; f < FC; ++f) acc[f] += part[f];
            } else if (act) {
#pragma unroll
                for (int f = 0; f < FC; ++f)
                    if (f < nf) {
                        float *q = A.out + ((int64_t)(f0 + f) * no + o) * A.np + p;
                        *q = (i0 == share.ibeg) ? part[f] : *q + part[f];
                    }
            }
        }
    }
}

// eight waves per SIMD (64 VGPRs, some scalars kept in vector lanes outside the
// inner loop) measured 793 -> 768 us against the compiler's own seven on
// 75 x 128 x 512 x 512, cubic
template <int GK, int SUM, int FC, bool GEOM, int MODE>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8))) void
k_das_wave(DasArgs A, WaveArgs W)
{
    extern __shared__ float sm[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nw = blockDim.x >> 6;
    uint32_t tile = blockIdx.x;
    int chunk = blockIdx.y, nchunk = gridDim.y;
    if (W.slab) {
        // each XCD takes every eighth outer element over all tiles: a channel's
        // row enters one L2 only
        chunk = tile & 7u;
        nchunk = 8;
        tile >>= 3;
    } else {
        // runs of `group` neighbouring tiles per XCD, dealt round robin: table
        // lines are shared in an L2, and every XCD gets shallow and deep tiles
        // (few and many receivers)
        const uint32_t g = W.group, s8 = tile >> 3;
        if (tile < gridDim.x / (8u * g) * (8u * g))
            tile = ((s8 / g) * 8u + (tile & 7u)) * g + s8 % g;
    }
    const int64_t i = (int64_t)tile * 64 + lane;
    const bool act = i < A.np;
    int64_t p = 0;
    if (act) {
        p = i;
        if (A.perm) {
            p = A.perm[i];
        } else if (W.fast) {
            const int fast = *W.fast;
            if (fast) p = band_pixel(i, A.np, fast);
        }
    }
    const int f0 = blockIdx.z * FC;
    const int nf = min(FC, A.nfr - f0);
    float pv[3] = {0.0f, 0.0f, 0.0f};
    if (GEOM) {
        // 2-D points run the 3-D geometry with zero third coordinates, which
        // adds exact zeros to its sums
        for (int d = 0; d < A.geo; ++d) {
            const float v = A.pvec[p * A.geo + d];
            if (d == 0) pv[0] = v;
            else if (d == 1) pv[1] = v;
            else pv[2] = v;
        }
    }
    const bool itx = W.inner_tx != 0;
    WaveShare share{0, itx ? A.ntx : A.nrx, W.split_inner ? chunk : chunk + nchunk * wave,
                    itx ? A.nrx : A.ntx, W.split_inner ? nchunk : nchunk * nw, ~0ull};
    if (W.split_inner) share.pat = every_nth(wave, nw);

    float acc[FC];
#pragma unroll
    for (int f = 0; f < FC; ++f) acc[f] = 0.0f;
    wave_sweep<GK, SUM, FC, GEOM, MODE>(A, W, sm, share, nw, wave, lane, act, p, pv, f0, nf, acc);
    if (SUM == WS_BOTH) {
        __syncthreads();
#pragma unroll
        for (int f = 0; f < FC; ++f) sm[(wave * FC + f) * 64 + lane] = acc[f];
        __syncthreads();
        if (wave < FC) {
            for (int f = wave; f < nf; f += min(nw, FC)) {
                float s = sm[f * 64 + lane];
                for (int v = 1; v < nw; ++v) s += sm[(v * FC + f) * 64 + lane];
                if (act) A.out[((int64_t)chunk * A.nfr + f0 + f) * A.np + p] = s;
            }
        }
    }
}

int wave_launch_sample(int gk, const DasArgs &a, const WaveArgs &w, int sum, int fc, int mode,
                       dim3 grid, int nw, size_t lds, hipStream_t s);
int wave_launch_cubic(const DasArgs &a, const WaveArgs &w, int sum, int fc, int mode, dim3 grid,
                      int nw, size_t lds, hipStream_t s);
int wave_launch_hermite(int gk, const DasArgs &a, const WaveArgs &w, int sum, int fc, int mode,
                        dim3 grid, int nw, size_t lds, hipStream_t s);

template <int GK, int SUM, int FC, bool GEOM>
static void wave_mode(int mode, const DasArgs &a, const WaveArgs &w, dim3 grid, int nw, size_t lds,
                      hipStream_t s)
{
    const dim3 block((unsigned)nw * 64);
    if (mode == WM_RECIP0)
        hipLaunchKernelGGL((k_das_wave<GK, SUM, FC, GEOM, WM_RECIP0>), grid, block, lds, s, a, w);
    else if (mode == WM_RECIP)
        hipLaunchKernelGGL((k_das_wave<GK, SUM, FC, GEOM, WM_RECIP>), grid, block, lds, s, a, w);
    else
        hipLaunchKernelGGL((k_das_wave<GK, SUM, FC, GEOM, WM_DIV>), grid, block, lds, s, a, w);
}

template <int GK, int SUM, int FC>
static void wave_geo(int mode, const DasArgs &a, const WaveArgs &w, dim3 grid, int nw, size_t lds,
                     hipStream_t s)
{
    if (a.geo)
        wave_mode<GK, SUM, FC, true>(mode, a, w, grid, nw, lds, s);
    else
        wave_mode<GK, SUM, FC, false>(mode, a, w, grid, nw, lds, s);
}

template <int GK, int SUM>
static void wave_fc(int fc, int mode, const DasArgs &a, const WaveArgs &w, dim3 grid, int nw,
                    size_t lds, hipStream_t s)
{
    if (fc == 4)
        wave_geo<GK, SUM, 4>(mode, a, w, grid, nw, lds, s);
    else if (fc == 2)
        wave_geo<GK, SUM, 2>(mode, a, w, grid, nw, lds, s);
    else
        wave_geo<GK, SUM, 1>(mode, a, w, grid, nw, lds, s);
}

template <int GK>
static int wave_sum(int sum, int fc, int mode, const DasArgs &a, const WaveArgs &w, dim3 grid,
                    int nw, size_t lds, hipStream_t s)
{
    if (sum == WS_BOTH)
        wave_fc<GK, WS_BOTH>(fc, mode, a, w, grid, nw, lds, s);
    else if (sum == WS_SEP)
        wave_fc<GK, WS_SEP>(fc, mode, a, w, grid, nw, lds, s);
    else
        wave_fc<GK, WS_NONE>(fc, mode, a, w, grid, nw, lds, s);
    return check_launch("das gather (wave tiles)");
}

}  // namespace pycbf
