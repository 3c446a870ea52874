// Ragged batches of Synthetic cubic DAS / SLSC requests in one persistent
// launch (no reference counterpart: pycbf beamforms one configuration per
// call, pycbf/gpu/__core_bf_classes__.py:68-118).
//
// A batch is a list of requests, each with its own plane-wave / element
// geometry (pycbf_synthetic_pack), x-major pixel grid, transmit / receive
// counts and output.  All requests share nt, so their channels are
// prefiltered by one launch of the natural-spline kernel over the
// concatenated channel data.  The gather is one persistent kernel: every
// workgroup pulls work items (request, TILE x TILE pixel tile, chunk of RC
// receive elements) from a queue ordered by cost (largest first) through one
// atomic counter, and exits when the queue is empty.  An item is walked in
// 8 x 8 pixel patches by the sweep of the wave-tile gather (das_wave.h): the
// transmits' delays once per patch in LDS, the chunk's receive elements split
// over the workgroup's waves, elements no pixel of the patch can use dropped.
// DAS requests add a patch's sum into the zeroed image with one float atomic
// per pixel; SLSC requests write per-receive images (every (receive element,
// pixel) is owned by one item), which the per-request SLSC launches then
// reduce.  64 requests of up to 75 x 256 channels x 4096: gather 14.4 -> 10.1 ms;
// 10 requests of about 31 x 128 x 2048 onto 256 x 256: 1.68 -> 0.85 ms (one wave
// per patch with 8 or 16 transmits in registers before).  Each item stamps its
// request's completion time (wall clock) for per-request latencies.
// Every launch of a run is a kernel (no memset), so a run can be captured in
// a graph.
#include <math.h>

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "das_wave.h"

namespace pycbf {

struct BatchReqDev {
    const float *txpack, *rxpack, *pvec;
    const float *coef;  // (ntx*nrx, nt+1) (y, e) pairs of this request
    float *out;         // DAS: (np); SLSC: per-receive images (nrx, np)
    int ntx, nrx, nx, nz, kind, nt;
    float c0, t0, dt, rdt, tmax, thresh;
};

struct BatchItem {
    int req, tile, r0, pad;
};

constexpr int BATCH_NW = 4;  // waves per workgroup

// One item: (tile / 8)^2 patches of 8 x 8 pixels, the receive elements
// r0 .. r0 + rchunk - 1, all transmits.
template <int KIND, int MODE>
__device__ __forceinline__ void batch_item(const BatchReqDev &R, const BatchItem &w, int tile,
                                           int rchunk, int ib, float *sm, int wave, int lane)
{
    constexpr int SUM = KIND == 0 ? WS_BOTH : WS_SEP;
    DasArgs A{};
    A.src = R.coef;
    A.ch_stride = 2 * ((int64_t)R.nt + 1);
    A.ntx = R.ntx;
    A.nrx = R.nrx;
    A.nfr = 1;
    A.np = (int64_t)R.nx * R.nz;
    A.nsrc = R.nt;
    A.t0 = R.t0;
    A.dt = R.dt;
    A.rdt = R.rdt;
    A.tmax = R.tmax;
    A.thresh = R.thresh;
    A.out = R.out;
    A.geo = 2;
    A.txpack = R.txpack;
    A.rxpack = R.rxpack;
    A.c0 = R.c0;
    WaveArgs W{};
    W.ib = ib;
    W.weights = !(R.thresh > 0.0f && R.thresh <= 1.0f);
    W.nhalf = (float)R.nt - 0.5f;
    const int r1 = min(w.r0 + rchunk, R.nrx);
    WaveShare share;
    // few transmits: the receive elements are the inner axis and the waves split them
    const bool few = KIND == 0 && R.ntx < 8;
    if (few) {
        share = WaveShare{w.r0, r1, 0, R.ntx, 1, every_nth(wave, BATCH_NW)};
    } else {
        W.inner_tx = 1;
        share = WaveShare{0, R.ntx, w.r0 + wave, r1, BATCH_NW, ~0ull};
    }
    const int tiles_z = (R.nz + tile - 1) / tile;
    const int px0 = (w.tile / tiles_z) * tile, pz0 = (w.tile % tiles_z) * tile;
#pragma unroll 1
    for (int ox = 0; ox < tile && px0 + ox < R.nx; ox += 8)
#pragma unroll 1
        for (int oz = 0; oz < tile && pz0 + oz < R.nz; oz += 8) {
            const int ix = px0 + ox + (lane >> 3), iz = pz0 + oz + (lane & 7);
            const bool act = ix < R.nx && iz < R.nz;
            const int64_t p = act ? (int64_t)ix * R.nz + iz : 0;
            const float pv[3] = {R.pvec[2 * p], R.pvec[2 * p + 1], 0.0f};
            float acc[1] = {0.0f};
            wave_sweep<GK_CUBIC, SUM, 1, true, MODE>(A, W, sm, share, BATCH_NW, wave, lane, act, p,
                                                     pv, 0, 1, acc);
            __syncthreads();  // the patch is done: LDS is free
            if (KIND == 0) {
                sm[wave * 64 + lane] = acc[0];
                __syncthreads();
                if (wave == 0 && act) {
                    float s = sm[lane];
                    for (int v = 1; v < BATCH_NW; ++v) s += sm[v * 64 + lane];
                    unsafeAtomicAdd(R.out + p, s);
                }
                __syncthreads();
            }
        }
}

template <int MODE>
__global__ __launch_bounds__(64 * BATCH_NW) void k_batch_das(const BatchReqDev *__restrict__ reqs,
                                                             const BatchItem *__restrict__ items,
                                                             int nitems, unsigned *counter,
                                                             unsigned long long *finish, int tile,
                                                             int rchunk, int ib)
{
    extern __shared__ float sm[];
    __shared__ int s_item;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (;;) {
        // Wave 0 pulls for the workgroup and passes the item through LDS.  Every
        // lane of it executes the atomic, lane 0 adding 1 and the others 0, and
        // the item index and the exit test are uniform by construction.  (Under
        // `if (threadIdx.x == 0)` the compiler joins the stamp below and this
        // pull into one branch of lane 0 across the loop's back edge, and parks
        // that lane outside the loop that the other lanes keep running on a
        // stale index.)
        if (wave == 0) {
            const unsigned v = atomicAdd(counter, lane == 0 ? 1u : 0u);
            s_item = (int)__builtin_amdgcn_readfirstlane(v);
        }
        __syncthreads();
        const int it = __builtin_amdgcn_readfirstlane(s_item);
        if (it >= nitems) break;
        const BatchItem w = items[it];
        const BatchReqDev R = reqs[w.req];
        if (R.kind == 0)
            batch_item<0, MODE>(R, w, tile, rchunk, ib, sm, wave, lane);
        else
            batch_item<1, MODE>(R, w, tile, rchunk, ib, sm, wave, lane);
        // the item ended with a barrier: all of it is done
        const unsigned long long now = (unsigned long long)wall_clock64();
        if (wave == 0) atomicMax(finish + w.req, lane == 0 ? now : 0ull);
        __syncthreads();  // s_item may be written again
    }
}

// clears the queue counter, the completion stamps and the DAS images, and
// records the batch start time
__global__ __launch_bounds__(256) void k_batch_reset(unsigned *counter, unsigned long long *finish,
                                                     int nreq, float *zero, int64_t nzero,
                                                     unsigned long long *start)
{
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (g == 0) {
        *counter = 0u;
        *start = (unsigned long long)wall_clock64();
    }
    if (g < nreq) finish[g] = 0ull;
    for (int64_t i = g; i < nzero; i += (int64_t)gridDim.x * 256) zero[i] = 0.0f;
}

__global__ void k_batch_stamp(unsigned long long *slot)
{
    if (threadIdx.x == 0) *slot = (unsigned long long)wall_clock64();
}

// ---------------------------------------------------------------- host side
struct BatchPlan {
    std::vector<pycbf_batch_req> reqs;
    std::vector<int64_t> ch_off;  // first channel of each request in the concatenation
    int64_t nch = 0, npix_das = 0;
    int nt = 0;
    int tile = 16, rchunk = 32;
    int nitems = 0, max_items = 0;
    int ib = 1, weights = 0, mode = WM_DIV;  // the gather's LDS block and quotient mode
    int blocks = 0;                          // resident workgroups of the gather (0: not asked yet)
    float *das_out_base = nullptr;  // DAS outputs are zeroed as one range when contiguous
};

static int64_t items_for(const std::vector<pycbf_batch_req> &reqs, int tile, int rchunk,
                         std::vector<BatchItem> *out)
{
    struct Cost {
        double c;
        BatchItem it;
    };
    std::vector<Cost> v;
    for (size_t r = 0; r < reqs.size(); ++r) {
        const pycbf_batch_req &q = reqs[r];
        const int tx = (q.nx + tile - 1) / tile, tz = (q.nz + tile - 1) / tile;
        for (int r0 = 0; r0 < q.nrx; r0 += rchunk)
            for (int t = 0; t < tx * tz; ++t) {
                const double c = (double)q.ntx * std::min(rchunk, q.nrx - r0) * tile * tile;
                if (out) v.push_back({c, BatchItem{(int)r, t, r0, 0}});
                else v.push_back({c, BatchItem{}});
            }
    }
    if (out) {
        std::stable_sort(v.begin(), v.end(), [](const Cost &a, const Cost &b) { return a.c > b.c; });
        out->clear();
        for (auto &c : v) out->push_back(c.it);
    }
    return (int64_t)v.size();
}

struct BatchLayout {
    size_t coef = 0, uscr = 0, reqs = 0, items = 0, ctrl = 0, total = 0;
};

static BatchLayout batch_layout(const BatchPlan &P)
{
    BatchLayout L;
    L.coef = align_up((size_t)P.nch * (size_t)(P.nt + 1) * 8, 256);
    L.uscr = spline_scratch_bytes(P.nch, P.nt);
    L.reqs = align_up(P.reqs.size() * sizeof(BatchReqDev), 256);
    L.items = align_up((size_t)P.max_items * sizeof(BatchItem), 256);
    L.ctrl = align_up(256 + (P.reqs.size() + 2) * 8, 256);
    L.total = L.coef + L.uscr + L.reqs + L.items + L.ctrl + 6 * 256;
    return L;
}

struct BatchPtrs {
    float2 *coef;
    float *uscr;
    BatchReqDev *reqs;
    BatchItem *items;
    unsigned *counter;
    unsigned long long *start, *finish;
};

static BatchPtrs carve(const BatchPlan &P, void *ws, size_t bytes)
{
    const BatchLayout L = batch_layout(P);
    Carver cv(ws, bytes);
    BatchPtrs b;
    b.coef = (float2 *)cv.take(L.coef);
    b.uscr = (float *)cv.take(L.uscr);
    b.reqs = (BatchReqDev *)cv.take(L.reqs);
    b.items = (BatchItem *)cv.take(L.items);
    char *ctrl = (char *)cv.take(L.ctrl);
    b.counter = (unsigned *)ctrl;
    b.start = (unsigned long long *)(ctrl + 256);
    b.finish = b.start + 1;
    return b;
}

// uploads the request table and the item list for (tile, rchunk)
static int upload(BatchPlan &P, const BatchPtrs &b, hipStream_t s)
{
    std::vector<BatchReqDev> dev(P.reqs.size());
    for (size_t r = 0; r < P.reqs.size(); ++r) {
        const pycbf_batch_req &q = P.reqs[r];
        BatchReqDev &d = dev[r];
        d.txpack = q.txpack;
        d.rxpack = q.rxpack;
        d.pvec = q.pvec;
        d.coef = (const float *)(b.coef + P.ch_off[r] * (int64_t)(P.nt + 1));
        d.out = q.kind == PYCBF_BATCH_DAS ? q.out : q.imrx;
        d.ntx = q.ntx;
        d.nrx = q.nrx;
        d.nx = q.nx;
        d.nz = q.nz;
        d.kind = q.kind == PYCBF_BATCH_DAS ? 0 : 1;
        d.nt = P.nt;
        d.c0 = q.c0;
        d.t0 = q.t0;
        d.dt = q.dt;
        d.rdt = 1.0f / q.dt;
        d.tmax = q.t0 + q.dt * (float)(P.nt - 1);
        d.thresh = q.thresh;
    }
    std::vector<BatchItem> items;
    P.nitems = (int)items_for(P.reqs, P.tile, P.rchunk, &items);
    if (int rc = check(hipMemcpyAsync(b.reqs, dev.data(), dev.size() * sizeof(BatchReqDev),
                                      hipMemcpyHostToDevice, s),
                       "batch request upload"))
        return rc;
    if (int rc = check(hipMemcpyAsync(b.items, items.data(), items.size() * sizeof(BatchItem),
                                      hipMemcpyHostToDevice, s),
                       "batch item upload"))
        return rc;
    // the host vectors go out of scope: wait for the copies
    return check(hipStreamSynchronize(s), "batch upload");
}

template <int MODE>
static int launch_gather_m(BatchPlan &P, const BatchPtrs &b, hipStream_t s)
{
    const size_t lds = std::max(wave_lds_bytes(P.ib, P.weights, BATCH_NW), (size_t)BATCH_NW * 256);
    if (!P.blocks) {
        // as many workgroups as can be resident at once, so that the queue is
        // drained by the full complement of waves
        int dev = 0, cus = 256, per_cu = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            cus <= 0)
            cus = 256;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_batch_das<MODE>,
                                                         64 * BATCH_NW, lds) != hipSuccess ||
            per_cu < 1)
            per_cu = 4;
        P.blocks = cus * per_cu;
    }
    hipLaunchKernelGGL(k_batch_das<MODE>, dim3(P.blocks), dim3(64 * BATCH_NW), lds, s, b.reqs,
                       b.items, P.nitems, b.counter, b.finish, P.tile, P.rchunk, P.ib);
    return check_launch("batch gather");
}

static int launch_gather(BatchPlan &P, const BatchPtrs &b, hipStream_t s)
{
    ProfScope ps("batch_gather", s);
    if (P.mode == WM_RECIP0) return launch_gather_m<WM_RECIP0>(P, b, s);
    if (P.mode == WM_RECIP) return launch_gather_m<WM_RECIP>(P, b, s);
    return launch_gather_m<WM_DIV>(P, b, s);
}

static int run_batch(BatchPlan &P, const float *rf_all, void *ws, size_t bytes, hipStream_t s,
                     bool gather_only)
{
    const BatchPtrs b = carve(P, ws, bytes);
    const int64_t nzero = P.das_out_base ? P.npix_das : 0;
    const int zb = (int)std::min<int64_t>(std::max<int64_t>((nzero + 255) / 256, 1), 4096);
    hipLaunchKernelGGL(k_batch_reset, dim3((unsigned)std::max<int64_t>(zb, (P.reqs.size() + 255) / 256)),
                       dim3(256), 0, s, b.counter, b.finish, (int)P.reqs.size(), P.das_out_base,
                       nzero, b.start);
    if (int rc = check_launch("batch reset")) return rc;
    if (!gather_only)
        if (int rc = launch_spline_coefs(rf_all, P.nch, P.nt, P.reqs[0].dt, b.uscr, b.coef, s))
            return rc;
    if (int rc = launch_gather(P, b, s)) return rc;
    if (gather_only) return 0;
    for (size_t r = 0; r < P.reqs.size(); ++r) {
        const pycbf_batch_req &q = P.reqs[r];
        if (q.kind != PYCBF_BATCH_SLSC) continue;
        if (int rc = launch_slsc(q.imrx, 1, q.nrx, q.nx, q.nz, q.sel, q.kwin, q.kofs, q.dsfx,
                                 q.dsfz, q.lags, q.nlag, q.precision, q.out, s))
            return rc;
        hipLaunchKernelGGL(k_batch_stamp, dim3(1), dim3(64), 0, s, b.finish + r);
        if (int rc = check_launch("batch stamp")) return rc;
    }
    return 0;
}

}  // namespace pycbf

using namespace pycbf;

struct pycbf_batch {
    BatchPlan plan;
};

extern "C" {

int pycbf_batch_create(const pycbf_batch_req *reqs, int nreq, pycbf_batch **out)
{
    if (!reqs || nreq < 1 || !out) return fail(PYCBF_EINVAL, "empty batch");
    BatchPlan P;
    P.nt = reqs[0].nt;
    int64_t chans = 0, das_pix = 0;
    float *das_next = nullptr;
    bool das_contig = true;
    for (int r = 0; r < nreq; ++r) {
        const pycbf_batch_req &q = reqs[r];
        if (q.kind != PYCBF_BATCH_DAS && q.kind != PYCBF_BATCH_SLSC)
            return fail(PYCBF_EINVAL, "request %d: kind %d", r, q.kind);
        if (q.ntx < 1 || q.nrx < 1 || q.nx < 1 || q.nz < 1 || q.nt != P.nt || q.nt < 1)
            return fail(PYCBF_EINVAL, "request %d: sizes (all requests share nt)", r);
        if (!q.txpack || !q.rxpack || !q.pvec || !q.out)
            return fail(PYCBF_EINVAL, "request %d: NULL pointer", r);
        if (!(q.dt > 0.0f) || q.dt != reqs[0].dt)
            return fail(PYCBF_EINVAL, "request %d: all requests share dt > 0", r);
        if (q.kind == PYCBF_BATCH_SLSC) {
            if (!q.imrx) return fail(PYCBF_EINVAL, "request %d: SLSC needs imrx scratch", r);
            if (q.nrx > 256 || q.kwin < 1 || q.kwin > 32 || q.kofs > 0 || q.kofs < -(q.kwin - 1) ||
                q.dsfx < 1 || q.dsfz < 1 || q.nlag < 1 || q.nlag > 64 ||
                q.precision < PYCBF_SLSC_FP32 || q.precision > PYCBF_SLSC_MFMA_BF16)
                return fail(PYCBF_EINVAL, "request %d: SLSC arguments", r);
            for (int i = 0; i < q.nlag; ++i)
                if (q.lags[i] < 1 || q.lags[i] > 63)
                    return fail(PYCBF_EINVAL, "request %d: lag out of range", r);
        } else {
            // DAS images are cleared by one range when they are laid out back to back
            if (das_next && q.out != das_next) das_contig = false;
            if (!P.das_out_base) P.das_out_base = q.out;
            das_next = q.out + (int64_t)q.nx * q.nz;
            das_pix += (int64_t)q.nx * q.nz;
        }
        P.ch_off.push_back(chans);
        chans += (int64_t)q.ntx * q.nrx;
        P.reqs.push_back(q);
        // No time lies on a trace whose start (or end) is no finite number, and the
        // gather's row offsets are formed from the quotient by dt: the request keeps
        // its zeros through a threshold that no weight reaches.
        const float tmax = q.t0 + q.dt * (float)(P.nt - 1);
        if (!std::isfinite(q.t0) || std::isnan(tmax)) {
            P.reqs.back().t0 = 0.0f;
            P.reqs.back().thresh = INFINITY;
        }
    }
    if (!das_contig)
        return fail(PYCBF_EINVAL, "DAS outputs must be contiguous, in request order");
    P.nch = chans;
    P.npix_das = das_pix;
    // One LDS block of inner elements for every request (the transmits, or a
    // receive chunk of a request with few of them), within 160 rows (weights
    // take a second array: 80), and one quotient mode that all of them allow.
    int inner = 1;
    P.mode = WM_RECIP0;
    for (const pycbf_batch_req &q : P.reqs) {
        inner = std::max(inner, q.kind == PYCBF_BATCH_DAS && q.ntx < 8 ? std::min(q.nrx, 128) : q.ntx);
        if (!(q.thresh > 0.0f && q.thresh <= 1.0f)) P.weights = 1;
        P.mode = std::min(P.mode, wave_mode_of(q.t0, q.dt, 1.0f / q.dt,
                                               q.t0 + q.dt * (float)(P.nt - 1), P.nt));
    }
    const int cap = P.weights ? 80 : 160, parts = (inner + cap - 1) / cap;
    P.ib = ((inner + parts - 1) / parts + 15) / 16 * 16;
    for (int t : {8, 16, 32})
        for (int c : {16, 32, 64, 128})
            P.max_items = (int)std::max<int64_t>(P.max_items, items_for(P.reqs, t, c, nullptr));
    *out = new pycbf_batch{P};
    return 0;
}

void pycbf_batch_destroy(pycbf_batch *b) { delete b; }

size_t pycbf_batch_workspace_bytes(const pycbf_batch *b)
{
    return b ? batch_layout(b->plan).total : 0;
}

int pycbf_batch_configure(pycbf_batch *b, int tile, int rchunk, void *workspace,
                          size_t workspace_bytes, void *stream)
{
    if (!b) return fail(PYCBF_EINVAL, "NULL batch");
    if ((tile != 8 && tile != 16 && tile != 32) ||
        (rchunk != 16 && rchunk != 32 && rchunk != 64 && rchunk != 128))
        return fail(PYCBF_EINVAL, "tile must be 8, 16 or 32 and rchunk 16, 32, 64 or 128");
    if (!workspace || workspace_bytes < batch_layout(b->plan).total)
        return fail(PYCBF_EINVAL, "workspace too small");
    b->plan.tile = tile;
    b->plan.rchunk = rchunk;
    return upload(b->plan, carve(b->plan, workspace, workspace_bytes), (hipStream_t)stream);
}

int pycbf_batch_run(pycbf_batch *b, const float *rf_all, void *workspace, size_t workspace_bytes,
                    void *stream)
{
    if (!b || !rf_all) return fail(PYCBF_EINVAL, "NULL argument");
    if (!workspace || workspace_bytes < batch_layout(b->plan).total)
        return fail(PYCBF_EINVAL, "workspace too small");
    if (b->plan.nitems == 0) return fail(PYCBF_EINVAL, "batch not configured");
    return run_batch(b->plan, rf_all, workspace, workspace_bytes, (hipStream_t)stream, false);
}

int pycbf_batch_autotune(pycbf_batch *b, const float *rf_all, int reps, void *workspace,
                         size_t workspace_bytes, void *stream, int *best_tile, int *best_rchunk,
                         float *times_ms)
{
    if (!b || !rf_all || reps < 1) return fail(PYCBF_EINVAL, "bad autotune arguments");
    hipStream_t s = (hipStream_t)stream;
    const int tiles[3] = {8, 16, 32}, chunks[4] = {16, 32, 64, 128};
    float best = 1e30f;
    int bt = 16, bc = 32;
    hipEvent_t e0, e1;
    if (int rc = check(hipEventCreate(&e0), "event")) return rc;
    if (int rc = check(hipEventCreate(&e1), "event")) return rc;
    int rc = pycbf_batch_configure(b, 16, 32, workspace, workspace_bytes, stream);
    if (!rc) rc = run_batch(b->plan, rf_all, workspace, workspace_bytes, s, false);  // tables
    for (int ti = 0; ti < 3 && !rc; ++ti)
        for (int ci = 0; ci < 4 && !rc; ++ci) {
            rc = pycbf_batch_configure(b, tiles[ti], chunks[ci], workspace, workspace_bytes, stream);
            if (rc) break;
            rc = run_batch(b->plan, rf_all, workspace, workspace_bytes, s, true);  // warm
            if (rc) break;
            hipEventRecord(e0, s);
            for (int k = 0; k < reps && !rc; ++k)
                rc = run_batch(b->plan, rf_all, workspace, workspace_bytes, s, true);
            hipEventRecord(e1, s);
            if (!rc) rc = check(hipEventSynchronize(e1), "autotune sync");
            float ms = 0.0f;
            hipEventElapsedTime(&ms, e0, e1);
            ms /= (float)reps;
            if (times_ms) times_ms[ti * 4 + ci] = ms;
            if (ms < best) {
                best = ms;
                bt = tiles[ti];
                bc = chunks[ci];
            }
        }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    if (rc) return rc;
    if (best_tile) *best_tile = bt;
    if (best_rchunk) *best_rchunk = bc;
    return pycbf_batch_configure(b, bt, bc, workspace, workspace_bytes, stream);
}

int pycbf_batch_latencies(const pycbf_batch *b, const void *workspace, size_t workspace_bytes,
                          double *latency_ms)
{
    if (!b || !workspace || !latency_ms) return fail(PYCBF_EINVAL, "NULL argument");
    const BatchPtrs p = carve(b->plan, const_cast<void *>(workspace), workspace_bytes);
    const size_t n = b->plan.reqs.size();
    std::vector<unsigned long long> v(n + 1);
    if (int rc = check(hipMemcpy(v.data(), p.start, (n + 1) * 8, hipMemcpyDeviceToHost),
                       "latency readback"))
        return rc;
    int dev = 0, khz = 0;
    hipGetDevice(&dev);
    if (int rc = check(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev),
                       "wall clock rate"))
        return rc;
    for (size_t r = 0; r < n; ++r)
        latency_ms[r] = (double)(long long)(v[r + 1] - v[0]) / (double)khz;
    return 0;
}

}  // extern "C"
