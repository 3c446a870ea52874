"""Ragged batches (pycbf_batch_*): every request of one persistent launch
against the single-request path, every autotuner configuration, and graph
replays against the eager run.

Bars: DAS images within 1e-5 of the single-request image's peak (float32
sums in another order); SLSC images (FP32) within 1e-4 absolute of SLSC on the
single-request per-receive images, NaN in the same places."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _requests(seed=0, nt=768):
    from pycbf_amd import sim
    from pycbf_amd.gpu.batch import BatchRequest
    rng = np.random.default_rng(seed)
    shapes = [(16, 24, 1, 8, "das"), (40, 33, 3, 16, "das"), (24, 24, 5, 24, "slsc"),
              (9, 70, 2, 12, "das"), (32, 16, 4, 40, "slsc"), (48, 40, 7, 20, "das"),
              # 136 receive elements: a ragged second chunk at every receive chunk
              (12, 10, 2, 136, "das")]
    reqs = []
    for k, (nx, nz, ntx, nrx, kind) in enumerate(shapes):
        xele = sim.linear_array(nrx)
        steers = np.radians(np.linspace(-10, 10, ntx)) if ntx > 1 else np.zeros(1)
        lim = float(xele[-1]) * 1.2 + 1e-3
        _, _, pnts = sim.grid(nx, nz, (-lim, lim), (2e-3, 14e-3))
        params = sim.pw_synthetic(steers, xele, pnts)
        xs, zs, amp = sim.scatterers(6, 60, (-lim, lim), (3e-3, 13e-3), seed + k)
        rf = sim.simulate_rf(steers, xele, nt, xs, zs, amp, seed=seed + k).astype(np.float32)
        reqs.append((BatchRequest(params=params, gridshape=(nx, nz), kind=kind,
                                  lags=tuple(range(1, 6)), kwin=4, dsfz=2, precision="fp32"),
                     rf))
    return reqs


def _single(req, rf, nt):
    """The same request through SyntheticBeamformer (+ slsc)."""
    import torch
    from pycbf_amd import sim
    from pycbf_amd.gpu import SyntheticBeamformer, slsc
    nx, nz = req.gridshape
    if req.kind == "das":
        bf = SyntheticBeamformer(**req.params, t0=0.0, dt=1.0 / sim.FS, nt=nt,
                                 interp={"kind": "cubic"}, sumtype="tx_and_rx")
        return bf(rf).reshape(nx, nz)
    bf = SyntheticBeamformer(**req.params, t0=0.0, dt=1.0 / sim.FS, nt=nt,
                             interp={"kind": "cubic"}, sumtype="tx_only")
    imrx = bf(rf, out_as_numpy=False)
    apod = bf.tables()[3]
    nrx = imrx.shape[0]
    return slsc(imrx.view(nrx, nx, nz), req.lags, req.kwin, -(req.kwin // 2),
                apod.view(nrx, nx, nz), req.dsfx, req.dsfz, "fp32").cpu().numpy()


def _check(batch, reqs, refs):
    for r, ((req, _), ref) in enumerate(zip(reqs, refs)):
        got = batch.outputs[r].cpu().numpy()
        assert got.shape == ref.shape, r
        if req.kind == "das":
            peak = np.max(np.abs(ref))
            assert np.max(np.abs(got - ref)) <= 1e-5 * peak, r
        else:
            assert np.array_equal(np.isnan(got), np.isnan(ref)), r
            fin = ~np.isnan(ref)
            assert np.max(np.abs(got[fin] - ref[fin])) <= 1e-4, r


@pytest.fixture(scope="module")
def setup():
    import torch
    from pycbf_amd import sim
    from pycbf_amd.gpu.batch import RaggedBatch
    nt = 768
    reqs = _requests(nt=nt)
    refs = [_single(q, rf, nt) for q, rf in reqs]
    batch = RaggedBatch([q for q, _ in reqs], nt=nt, dt=1.0 / sim.FS)
    for v, (_, rf) in zip(batch.rf_views, reqs):
        v.copy_(torch.as_tensor(rf))
    return batch, reqs, refs


def test_batch_matches_single_requests(setup):
    import torch
    batch, reqs, refs = setup
    print("ragged batch of 7 requests, default configuration", flush=True)
    batch.run()
    torch.cuda.synchronize()
    _check(batch, reqs, refs)
    lat = batch.latencies_ms()
    assert np.all(lat > 0) and np.all(np.isfinite(lat))


@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("rchunk", [16, 32, 64, 128])
def test_batch_every_configuration(setup, tile, rchunk):
    import torch
    batch, reqs, refs = setup
    print(f"ragged batch tile {tile} rchunk {rchunk}", flush=True)
    batch.configure(tile, rchunk)
    batch.run()
    torch.cuda.synchronize()
    _check(batch, reqs, refs)


def test_autotune_then_graph_replays(setup):
    import torch
    batch, reqs, refs = setup
    tile, rchunk, times = batch.autotune(reps=1)
    assert (tile, rchunk) in times and times[(tile, rchunk)] == min(times.values())
    batch.run()
    torch.cuda.synchronize()
    eager = [o.clone() for o in batch.outputs]
    batch.capture()
    for k in range(3):
        for o in batch.outputs:      # the program's own eager work between replays
            o.fill_(-7.0) if o.dtype == torch.float32 else None
        torch.cuda.synchronize()
        batch.run()
        torch.cuda.synchronize()
        for r, (o, e) in enumerate(zip(batch.outputs, eager)):
            assert torch.equal(torch.isnan(o), torch.isnan(e)), (k, r)
            ok = ~torch.isnan(e)
            assert float((o[ok] - e[ok]).abs().max()) <= 1e-5 * float(e[ok].abs().max() + 1e-30), (k, r)
    _check(batch, reqs, refs)


@pytest.mark.parametrize("t0", [0.0, 1.5e-6])
@pytest.mark.parametrize("thresh", [0.0, 1e-2, 1.5])
def test_batch_gather_branches(t0, thresh):
    """Few transmits (the waves split the receive elements), more transmits than
    one LDS block, grids smaller than a patch and with ragged edges, thresholds
    where zero weights count (0) and where nothing does (1.5), and a trace
    start away from zero, against the single-request beamformer (1e-5 of the
    peak, summation order)."""
    import torch
    from pycbf_amd import sim
    from pycbf_amd.gpu import SyntheticBeamformer
    from pycbf_amd.gpu.batch import BatchRequest, RaggedBatch
    nt, dt = 500, 1.0 / sim.FS
    rng = np.random.default_rng(3)
    reqs, singles = [], []
    for ntx, nrx, nx, nz in ((1, 20, 5, 7), (7, 130, 9, 17), (8, 9, 33, 8), (170, 3, 16, 21)):
        xele = sim.linear_array(nrx)
        _, _, pnts = sim.grid(nx, nz, (-2e-3, 2e-3), (2e-3, 7e-3))
        p = sim.pw_synthetic(np.radians(np.linspace(-9, 9, ntx)) if ntx > 1 else np.zeros(1), xele, pnts)
        reqs.append(BatchRequest(params=p, gridshape=(nx, nz), thresh=thresh))
        singles.append(SyntheticBeamformer(**p, t0=t0, dt=dt, nt=nt, interp={"kind": "cubic"}, thresh=thresh))
    batch = RaggedBatch(reqs, nt=nt, dt=dt, t0=t0)
    for v in batch.rf_views:
        v.copy_(torch.as_tensor(rng.standard_normal(tuple(v.shape)).astype(np.float32)))
    for tile, rchunk in ((8, 16), (16, 128), (32, 32)):
        batch.configure(tile, rchunk)
        batch.run()
        for bf, v, o in zip(singles, batch.rf_views, batch.outputs):
            ref = bf(v, out_as_numpy=False).reshape(o.shape)
            assert float((o - ref).abs().max()) <= 1e-5 * float(ref.abs().max()), (tile, rchunk, tuple(o.shape))


@pytest.mark.parametrize("t0", [float("nan"), float("inf"), -float("inf")])
def test_batch_without_a_finite_trace_start(t0):
    """No time lies on a trace that starts nowhere: zero images, from few and
    from many transmits."""
    import torch
    from pycbf_amd import sim
    from pycbf_amd.gpu.batch import BatchRequest, RaggedBatch
    reqs = []
    for ntx, nrx, nx, nz in ((2, 20, 5, 7), (9, 8, 12, 9)):
        _, _, pnts = sim.grid(nx, nz, (-2e-3, 2e-3), (2e-3, 7e-3))
        p = sim.pw_synthetic(np.radians(np.linspace(-9, 9, ntx)), sim.linear_array(nrx), pnts)
        reqs.append(BatchRequest(params=p, gridshape=(nx, nz)))
    print(f"ragged batch t0={t0}", flush=True)
    batch = RaggedBatch(reqs, nt=500, dt=1.0 / sim.FS, t0=t0)
    batch.rf_all.normal_()
    batch.run()
    torch.cuda.synchronize()
    assert not any(bool(o.any()) for o in batch.outputs)


def test_batch_with_divisions():
    """Half a nanosecond per sample, below the steps whose reciprocal is tried:
    quotients by division, few and many transmits, against the oracle's Tabbed DAS
    on the geometry's own tables (1e-5 of the peak)."""
    import torch
    import oracle
    from pycbf_amd import sim
    from pycbf_amd.gpu import SyntheticBeamformer
    from pycbf_amd.gpu.batch import BatchRequest, RaggedBatch
    dt, nt, f = 5e-10, 500, 5e-10 * sim.FS  # positions scale with the step
    reqs, tabs = [], []
    for ntx, nrx, nx, nz in ((2, 20, 5, 7), (9, 8, 12, 9)):
        _, _, pnts = sim.grid(nx, nz, (-2e-3 * f, 2e-3 * f), (2e-3 * f, 7e-3 * f))
        p = sim.pw_synthetic(np.radians(np.linspace(-9, 9, ntx)), sim.linear_array(nrx) * f, pnts)
        reqs.append(BatchRequest(params=p, gridshape=(nx, nz)))
        bf = SyntheticBeamformer(**p, t0=0.0, dt=dt, nt=nt, interp={"kind": "cubic"})
        tabs.append([t.cpu().numpy() for t in bf.tables()])
    batch = RaggedBatch(reqs, nt=nt, dt=dt)
    batch.rf_all.normal_()
    print("ragged batch with divisions", flush=True)
    batch.run()
    torch.cuda.synchronize()
    for t, v, o in zip(tabs, batch.rf_views, batch.outputs):
        ref = oracle.das_tabbed(v.cpu().numpy(), 0.0, dt, *t, kind="cubic").reshape(o.shape)
        assert np.abs(ref).max() > 0
        assert np.abs(o.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()
