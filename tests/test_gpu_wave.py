"""The wave-tile gather (one frame of every kind, several frames of all but the
cubic) at the sizes where its tiling can go wrong, against the CPU oracle:
partial and single 64-pixel tiles, few transmits (the waves split the
receivers), inner axes over one LDS block, two and three frames, passes of
four with a remainder, a trace start away from zero, weights other than one,
delays off the trace and NaN.  Bar: 1e-5 of the image peak, as for every image
(per-sample outputs of nearest and linear bitwise)."""
import numpy as np
import pytest

import oracle
from oracle import numerics
from pycbf_amd import sim
from pycbf_amd.gpu import SyntheticBeamformer, TabbedBeamformer
from tests.helpers import assert_close_to_peak

pytestmark = pytest.mark.gpu

DT = 1.0 / 40e6
KINDS = [({"kind": "nearest"}, 1), ({"kind": "nearest", "usf": 3}, 3), ({"kind": "linear"}, 1),
         ({"kind": "cubic"}, 1), ({"kind": "korder_cubic", "k": 8}, 1), ({"kind": "makima"}, 1)]
# ntx, nrx, np, nfr, t0, unit transmit weights
SIZES = [(1, 5, 1, None, 0.0, True), (3, 33, 63, 2, 2e-6, False), (7, 16, 64, 3, 0.0, True),
         (8, 9, 65, None, -1e-6, False), (11, 20, 200, 5, 0.0, True), (170, 6, 130, None, 0.0, True),
         (90, 3, 70, 4, 1e-6, False), (2, 200, 129, None, 0.0, False)]


def _tables(ntx, nrx, npx, nt, t0, unit, rng):
    span = nt * DT
    tautx = (t0 + rng.uniform(0.0, 0.5, (ntx, npx)) * span).astype(np.float32)
    taurx = (rng.uniform(-0.05, 0.6, (nrx, npx)) * span).astype(np.float32)
    apodtx = np.ones((ntx, npx), np.float32) if unit else rng.uniform(0, 1, (ntx, npx)).astype(np.float32)
    apodrx = (rng.uniform(0, 1, (nrx, npx)) * (rng.random((nrx, npx)) < 0.7)).astype(np.float32)
    apodrx[:, ::5] = 0.0  # pixels that no receiver uses
    taurx[nrx // 2, ::3] = np.nan
    return tautx, apodtx, taurx, apodrx


def _reference(rf, t0, tabs, interp, usf, sumtype, monkeypatch):
    if interp["kind"] == "makima":
        # the C oracle has no makima: the thread-per-sample kernel, which places
        # and evaluates each sample with the same float32 operations
        monkeypatch.setenv("PYCBF_DAS_PLAIN", "1")
        out = _beamformer(tabs, t0, rf.shape[-1], interp, sumtype)(rf)
        monkeypatch.delenv("PYCBF_DAS_PLAIN")
        return out
    S = numerics.make_S(8).astype(np.float32) if interp["kind"] == "korder_cubic" else None
    return np.stack([oracle.das_tabbed(r, t0, DT, *tabs, kind=interp["kind"], usf=usf, sumtype=sumtype, S=S)
                     for r in rf])


def _beamformer(tabs, t0, nt, interp, sumtype):
    return TabbedBeamformer(tautx=tabs[0], apodtx=tabs[1], taurx=tabs[2], apodrx=tabs[3], t0=t0, dt=DT, nt=nt,
                            interp=interp, sumtype=sumtype)


@pytest.mark.parametrize("interp,usf", KINDS, ids=[k[0]["kind"] + str(k[1]) for k in KINDS])
@pytest.mark.parametrize("ntx,nrx,npx,nfr,t0,unit", SIZES)
def test_wave_gather_matches_oracle(ntx, nrx, npx, nfr, t0, unit, interp, usf, monkeypatch):
    rng = np.random.default_rng(ntx * 1000 + npx)
    nt = 120
    tabs = _tables(ntx, nrx, npx, nt, t0, unit, rng)
    rf = rng.standard_normal((nfr or 1, ntx, nrx, nt)).astype(np.float32)
    for sumtype in ("tx_and_rx", "tx_only", "rx_only", "none"):
        print(f"wave {interp} {ntx}x{nrx} {npx} px nfr={nfr} {sumtype}", flush=True)
        got = _beamformer(tabs, t0, nt, interp, sumtype)(rf if nfr else rf[0])
        ref = _reference(rf, t0, tabs, interp, usf, sumtype, monkeypatch)
        ref = ref if nfr else ref[0]
        if sumtype == "none" and interp["kind"] in ("nearest", "linear") and usf == 1:
            assert np.array_equal(got, ref.reshape(got.shape))
        else:
            assert_close_to_peak(got, ref.reshape(got.shape), 1e-5, sumtype)


def _last_quotient(t0, nt, usf):
    """(tmax - t0) / dt of the (upsampled) trace in float32, and its entries."""
    f = np.float32
    t0, dt = f(t0), f(DT)
    return float((f(t0 + dt * f(nt - 1)) - t0) / f(dt / f(usf))), usf * (nt - 1) + 1


@pytest.mark.parametrize("nfr", [None, 4])
@pytest.mark.parametrize("t0,nt,usf,past", [(0.5, 60, 1, 0.5), (0.5, 69, 1, 1.0), (0.05, 500, 16, 0.5)])
def test_nearest_at_a_last_sample_time_that_rounds_past_the_trace(t0, nt, usf, past, nfr):
    """A start so late that float32 moves the last sample time up by half a
    sample (past 0.5: the reciprocal quotients) or a whole one (past 1: the
    division): a delay there, in waves that lie on the trace as a whole, selects
    no sample.  Nearest picks samples, so the bar is the sum's own rounding."""
    q, n = _last_quotient(t0, nt, usf)
    assert n - 1 + past <= q < n - 0.5 + past
    rng = np.random.default_rng(nt)
    ntx, nrx, npx = 9, 10, 130
    last = np.float32(t0) + np.float32(DT) * np.float32(nt - 1)
    tautx = np.repeat(np.linspace(t0, last, npx, dtype=np.float32)[None], ntx, axis=0)
    tautx[:, ::4] = last
    assert tautx.min() >= np.float32(t0) and tautx.max() == last
    tabs = (tautx, np.ones((ntx, npx), np.float32), np.zeros((nrx, npx), np.float32),
            np.ones((nrx, npx), np.float32))
    rf = rng.standard_normal((nfr or 1, ntx, nrx, nt)).astype(np.float32)
    for sumtype in ("tx_and_rx", "tx_only", "rx_only"):
        print(f"late nearest t0={t0} nt={nt} usf={usf} nfr={nfr} {sumtype}", flush=True)
        got = _beamformer(tabs, t0, nt, {"kind": "nearest", "usf": usf}, sumtype)(rf if nfr else rf[0])
        ref = oracle.das_tabbed(rf if nfr else rf[0], t0, DT, *tabs, kind="nearest", usf=usf, sumtype=sumtype)
        assert not ref[..., ::4].any()
        assert_close_to_peak(got, ref, 1e-5, sumtype)


@pytest.mark.parametrize("interp", [{"kind": "cubic"}, {"kind": "linear"}, {"kind": "korder_cubic", "k": 8}],
                         ids=lambda i: i["kind"])
@pytest.mark.parametrize("ntx", [3, 9])
@pytest.mark.parametrize("on", ["tx", "rx"])
def test_infinite_weights_on_one_axis(on, ntx, interp, monkeypatch):
    """Weights of one on one axis and infinite ones on the other, where no sample
    lies on the trace (nothing is added) and where some do (infinite, or NaN where
    the signs differ): the infinities, NaN and finite pixels of the kernel that
    adds each sample by itself."""
    rng = np.random.default_rng(8)
    nrx, npx, nt = 12, 140, 200
    span = np.float32(nt * DT)
    tau = {"tx": rng.uniform(0, 0.4, (ntx, npx)).astype(np.float32) * span,
           "rx": rng.uniform(0, 0.4, (nrx, npx)).astype(np.float32) * span}
    apod = {"tx": np.ones((ntx, npx), np.float32), "rx": np.ones((nrx, npx), np.float32)}
    apod[on][1, ::7] = np.inf
    tau[on][1, ::7] += 2 * span   # off the trace
    apod[on][2, 3::7] = np.inf    # on it
    tabs = (tau["tx"], apod["tx"], tau["rx"], apod["rx"])
    rf = rng.standard_normal((ntx, nrx, nt)).astype(np.float32)
    for sumtype in ("tx_and_rx", "tx_only", "rx_only"):
        print(f"infinite {on} weights ntx={ntx} {interp['kind']} {sumtype}", flush=True)
        got = _beamformer(tabs, 0.0, nt, interp, sumtype)(rf)
        monkeypatch.setenv("PYCBF_DAS_PLAIN", "1")
        ref = _beamformer(tabs, 0.0, nt, interp, sumtype)(rf)
        monkeypatch.delenv("PYCBF_DAS_PLAIN")
        fin = np.isfinite(ref)
        assert fin[..., ::7].all() and not fin.all()
        assert np.array_equal(got[~fin], ref[~fin], equal_nan=True)
        assert np.isfinite(got[fin]).all()
        assert_close_to_peak(got[fin], ref[fin], 1e-5, sumtype)


@pytest.mark.parametrize("thresh", [0.0, 1e-2, 1.5])
@pytest.mark.parametrize("nfr", [None, 4])
@pytest.mark.parametrize("kind", ["cubic", "korder_cubic"])
def test_wave_gather_geometry_equals_its_tables(kind, nfr, thresh):
    """The point geometry and its own tables select the same samples, at
    thresholds where zero weights count (0), do not (0.01) and nothing does."""
    xele = sim.linear_array(24)
    _, _, pnts = sim.grid(9, 37, (-4e-3, 4e-3), (2e-3, 9e-3))
    p = sim.pw_synthetic(np.radians(np.linspace(-10, 10, 9)), xele, pnts)
    rf = np.random.default_rng(4).standard_normal((nfr or 1, 9, 24, 600)).astype(np.float32)
    rf = rf if nfr else rf[0]
    kw = dict(t0=0.0, dt=DT, nt=600, interp={"kind": kind}, thresh=thresh)
    syn = SyntheticBeamformer(**p, **kw)
    t = syn.tables()
    tab = TabbedBeamformer(tautx=t[0], apodtx=t[1], taurx=t[2], apodrx=t[3], **kw)
    a, b = syn(rf), tab(rf)
    assert_close_to_peak(a, b, 1e-6, f"{kind} thresh={thresh}")
    assert (thresh > 1.0) == (not np.any(b))


# which order and kernel a call over several frames takes: chunks of the outer axis
# per XCD (few tiles; per-sample outputs of a geometry; one transmit, 13 frames and
# more), finer chunks of it (few or many outer elements, small tables), and the
# staged gather (nearest, 9 frames of a table over 96 MB)
@pytest.mark.parametrize("ntx,nrx,nx,nz,nt,nfr,kind,sumtype,geo", [
    (9, 20, 12, 25, 300, 5, "linear", "none", True), (9, 20, 12, 25, 300, 5, "linear", "none", False),
    (1, 24, 65, 65, 300, 13, "nearest", "tx_only", True), (1, 24, 65, 65, 300, 12, "nearest", "tx_only", True),
    (3, 20, 10, 21, 300, 4, "linear", "rx_only", True), (17, 20, 10, 21, 300, 4, "korder_cubic", "rx_only", False),
    (9, 40, 65, 65, 300, 6, "linear", "tx_and_rx", True), (9, 15, 30, 30, 300, 4, "korder_cubic", "tx_and_rx", False),
    (9, 40, 20, 30, 300, 8, "nearest", "tx_and_rx", False), (50, 64, 97, 85, 2000, 9, "nearest", "tx_and_rx", True)])
def test_frame_batches_in_every_order(ntx, nrx, nx, nz, nt, nfr, kind, sumtype, geo, monkeypatch):
    """Every order of a frame batch against the kernel that adds each sample by
    itself; 1e-5 of the image peak (summation order)."""
    _, _, pnts = sim.grid(nx, nz, (-4e-3, 4e-3), (2e-3, 0.9 * nt * DT * sim.C0 / 2))
    steers = np.radians(np.linspace(-8, 8, ntx)) if ntx > 1 else np.zeros(1)
    kw = dict(t0=0.0, dt=DT, nt=nt, interp={"kind": kind}, sumtype=sumtype)
    if kind == "korder_cubic":
        kw["interp"]["k"] = 8
    bf = SyntheticBeamformer(**sim.pw_synthetic(steers, sim.linear_array(nrx), pnts), **kw)
    if not geo:
        t = bf.tables()
        bf = TabbedBeamformer(tautx=t[0], apodtx=t[1], taurx=t[2], apodrx=t[3], **kw)
    rf = np.random.default_rng(ntx + nt).standard_normal((nfr, ntx, nrx, nt)).astype(np.float32)
    print(f"batch {ntx}x{nrx}x{nt} {nx * nz} px nfr={nfr} {kind} {sumtype} geo={geo}", flush=True)
    got = bf(rf)
    monkeypatch.setenv("PYCBF_DAS_PLAIN", "1")
    assert_close_to_peak(got, bf(rf), 1e-5, sumtype)


@pytest.mark.parametrize("interp,usf", KINDS, ids=[k[0]["kind"] + str(k[1]) for k in KINDS])
@pytest.mark.parametrize("ntx,nrx,npx,nfr,t0", [(3, 12, 70, None, 0.0), (9, 10, 130, 5, 3e-8), (9, 10, 130, 2, 0.0)])
def test_wave_gather_with_divisions(ntx, nrx, npx, nfr, t0, interp, usf, monkeypatch):
    """Half a nanosecond per sample, below the steps whose reciprocal is tried
    (2^-30): quotients by division, integer row offsets.  Bars as above."""
    dt, nt = 5e-10, 120
    rng = np.random.default_rng(ntx + npx)
    tabs = list(_tables(ntx, nrx, npx, nt, 0.0, False, rng))
    tabs[0] = (tabs[0] * np.float32(dt / DT) + np.float32(t0)).astype(np.float32)
    tabs[2] = (tabs[2] * np.float32(dt / DT)).astype(np.float32)
    rf = rng.standard_normal((nfr or 1, ntx, nrx, nt)).astype(np.float32)
    monkeypatch.setitem(globals(), "DT", dt)  # of the oracle and the beamformers here
    for sumtype in ("tx_and_rx", "tx_only", "rx_only", "none"):
        print(f"divisions {interp} {ntx}x{nrx} nfr={nfr} {sumtype}", flush=True)
        got = _beamformer(tabs, t0, nt, interp, sumtype)(rf if nfr else rf[0])
        ref = _reference(rf, t0, tabs, interp, usf, sumtype, monkeypatch).reshape(got.shape)
        if sumtype == "none" and interp["kind"] in ("nearest", "linear") and usf == 1:
            assert np.array_equal(got, ref)
        else:
            assert_close_to_peak(got, ref, 1e-5, sumtype)


@pytest.mark.parametrize("kind", ["linear", "cubic", "korder_cubic", "akima"])
@pytest.mark.parametrize("nt", [60, 69])
def test_last_sample_time_past_the_last_knot(nt, kind, monkeypatch):
    """The late starts of the nearest test: at 69 samples the last time lies a
    whole sample past the last knot, whose index is clamped.  Against the kernel
    that places each sample by itself."""
    t0 = 0.5
    rng = np.random.default_rng(nt)
    last = np.float32(t0) + np.float32(DT) * np.float32(nt - 1)
    tautx = np.linspace(t0, last, 70, dtype=np.float32)[None].repeat(9, axis=0)
    tautx[:, ::4] = last
    tabs = (tautx, np.ones_like(tautx), np.zeros((4, 70), np.float32), np.ones((4, 70), np.float32))
    rf = rng.standard_normal((9, 4, nt)).astype(np.float32)
    interp = {"kind": kind, "k": 8} if kind == "korder_cubic" else {"kind": kind}
    for sumtype in ("tx_and_rx", "tx_only", "none"):
        got = _beamformer(tabs, t0, nt, interp, sumtype)(rf)
        monkeypatch.setenv("PYCBF_DAS_PLAIN", "1")
        ref = _beamformer(tabs, t0, nt, interp, sumtype)(rf)
        monkeypatch.delenv("PYCBF_DAS_PLAIN")
        assert_close_to_peak(got, ref, 1e-5, sumtype)


@pytest.mark.parametrize("interp,usf", [k for k in KINDS if k[0]["kind"] != "makima" and k[1] == 1],
                         ids=lambda v: v["kind"] if isinstance(v, dict) else "")
@pytest.mark.parametrize("nt", [2 ** 19, 2 ** 19 + 1])
def test_longest_float_offsets(nt, interp, usf, monkeypatch):
    """Traces at and one past the entries whose byte offsets a float's low bits
    hold, with delays among the last samples and at the last."""
    rng = np.random.default_rng(nt)
    last = np.float32(DT) * np.float32(nt - 1)
    tautx = rng.uniform(0, last, (1, 130)).astype(np.float32)
    tautx[0, 1::3] = last - (rng.uniform(0, 50, 43) * DT).astype(np.float32)
    tautx[0, ::3] = last
    tabs = (tautx, np.ones_like(tautx), np.zeros((2, 130), np.float32), np.ones((2, 130), np.float32))
    rf = rng.standard_normal((1, 1, 2, nt)).astype(np.float32)
    print(f"{nt} samples {interp}", flush=True)
    for sumtype in ("tx_and_rx", "none"):
        got = _beamformer(tabs, 0.0, nt, interp, sumtype)(rf[0])
        assert_close_to_peak(got, _reference(rf, 0.0, tabs, interp, usf, sumtype, monkeypatch)[0], 1e-5, sumtype)


@pytest.mark.parametrize("nfr", [None, 3, 9])
def test_direct_gather_by_its_own_order(nfr, monkeypatch):
    """PYCBF_DAS_LDS=0 selects the direct gather for every call: with unit weights
    its sums are the per-sample values added one after the other, receivers (per
    transmit) first, the transmits' sums then in order, bit for bit."""
    rng = np.random.default_rng(11)
    ntx, nrx, npx, nt = 5, 9, 300, 200
    tabs = [(rng.uniform(0, 0.4, (n, npx)) * nt * DT).astype(np.float32) for n in (ntx, nrx)]
    tabs = (tabs[0], np.ones((ntx, npx), np.float32), tabs[1], np.ones((nrx, npx), np.float32))
    rf = rng.standard_normal((nfr or 1, ntx, nrx, nt)).astype(np.float32)
    s = np.stack([oracle.das_tabbed(r, 0.0, DT, *tabs, kind="linear", sumtype="none") for r in rf])
    add = lambda x, axis: np.add.accumulate(x, axis=axis, dtype=np.float32).take(-1, axis=axis)  # noqa: E731
    per_tx = add(s, 2)
    ref = {"tx_and_rx": add(per_tx, 1), "tx_only": add(s, 1), "rx_only": per_tx, "none": s}
    monkeypatch.setenv("PYCBF_DAS_LDS", "0")
    for sumtype, want in ref.items():
        print(f"direct gather nfr={nfr} {sumtype}", flush=True)
        got = _beamformer(tabs, 0.0, nt, {"kind": "linear"}, sumtype)(rf if nfr else rf[0])
        assert np.array_equal(got, want if nfr else want[0]), sumtype


def test_direct_gather_of_a_geometry(monkeypatch):
    """The same switch over a point geometry: its delay tables, bit for bit."""
    p = sim.pw_synthetic(np.radians(np.linspace(-10, 10, 4)), sim.linear_array(12),
                         sim.grid(9, 37, (-4e-3, 4e-3), (2e-3, 9e-3))[2])
    rf = np.random.default_rng(4).standard_normal((2, 4, 12, 600)).astype(np.float32)
    monkeypatch.setenv("PYCBF_DAS_LDS", "0")
    for kind in ("nearest", "cubic", "korder_cubic"):
        kw = dict(t0=0.0, dt=DT, nt=600, interp={"kind": kind})
        syn = SyntheticBeamformer(**p, **kw)
        t = syn.tables()
        tab = TabbedBeamformer(tautx=t[0], apodtx=t[1], taurx=t[2], apodrx=t[3], **kw)
        assert np.array_equal(syn(rf), tab(rf)) and syn(rf).any(), kind


@pytest.mark.parametrize("nx,nz,xfast", [(13, 320, False), (64, 64, False), (37, 200, True), (4099, 1, False)])
def test_wave_gather_over_grids_in_their_own_order(nx, nz, xfast):
    """Tables handed over in the pixels' own order (das_tabbed): grids of z or
    x lines, a last band of fewer than eight lines, and pixels that form no
    grid (a prime count along one line)."""
    import torch
    from pycbf_amd.gpu.autograd import das_tabbed
    xele = sim.linear_array(16)
    _, _, pnts = sim.grid(nx, nz, (-3e-3, 3e-3), (3e-3, 9e-3))
    if xfast:
        pnts = np.ascontiguousarray(pnts.reshape(nx, nz, 2).transpose(1, 0, 2).reshape(-1, 2))
    tabs = sim.pw_tabs(np.radians([-6.0, 0.0, 4.0]), xele, pnts)
    rf = np.random.default_rng(9).standard_normal((3, 16, 700)).astype(np.float32)
    d = lambda a: torch.as_tensor(a, device="cuda")  # noqa: E731
    for kind in ("cubic", "linear"):
        got = das_tabbed(d(rf), *(d(t) for t in tabs), 0.0, DT, kind, "tx_and_rx", 1e-2).cpu().numpy()
        assert_close_to_peak(got, oracle.das_tabbed(rf, 0.0, DT, *tabs, kind=kind), 1e-5, kind)


@pytest.mark.parametrize("data", ["normal", "bursts"])
@pytest.mark.parametrize("nt", [4097, 8191, 8192, 8193, 16385, 32768, 32769])
def test_spline_prefilter_over_several_waves_bitwise(nt, data):
    """Channels shared by two to eight waves (and one sample past the longest),
    dense data and bursts between zero runs of up to 200 samples (guessed
    carries that have to be recomputed across a wave's edge): second
    derivatives bit for bit the reference recurrence's."""
    import torch
    from pycbf_amd.gpu import _engine as E
    rng = np.random.default_rng(nt)
    nch, dt = 5, np.float32(2.5e-8)
    rf = rng.standard_normal((nch, nt)).astype(np.float32)
    if data == "bursts":
        on = np.zeros((nch, nt), bool)
        for c in range(nch):
            k = 0
            while k < nt:
                n = int(rng.integers(1, 8))
                on[c, k:k + n] = True
                k += n + int(rng.integers(1, 200))
        rf *= on
    x = torch.as_tensor(rf, device="cuda")
    wsb = E.lib.pycbf_spline_workspace_bytes(nch, nt)
    ws = torch.empty(wsb, dtype=torch.uint8, device="cuda")
    y2 = torch.empty((nch, nt), dtype=torch.float32, device="cuda")
    E.check(E.lib.pycbf_spline_y2(E.ptr(x), nch, nt, float(dt), E.ptr(y2), E.ptr(ws), wsb, E.stream_of(x.device)), "y2")
    ref = np.stack([oracle.spline_y2(r, dt) for r in rf])
    assert np.array_equal(y2.cpu().numpy().view(np.uint32), ref.view(np.uint32))
