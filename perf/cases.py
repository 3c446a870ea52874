"""The work whose speed this repository keeps an eye on: beamforming calls as a program makes them, from one
small live frame to a batch of full compound frames, the coherence and multiply-and-sum beamformers, the
differentiable forms with their gradients, IQ demodulation and a ragged batch.

`listed()` gives the fixed cases, `draw(rng)` one more of the same ranges, `prepare(case, seed)` what a program
holds before the call, `run(state)` one pass through the public entry points, `work(case)` the bytes and
operations a pass cannot do without, and `exact(case, seed)` the same outputs in 64 bits from plain torch.
"""
import math

import numpy as np
import torch

FS, FC, C0 = 40e6, 5e6, 1540.0
DT = float(np.float32(1.0 / FS))  # the engines take the sample spacing as a float32
PITCH = 0.3e-3
FNUM = 1.5
THRESH = 1e-2                     # the beamformers' own default
SLSC_LAGS, SLSC_KWIN = tuple(range(1, 21)), 8


def listed():
    """Sizes are those of the benchmark and the tests, or ordinary ones of a 64 .. 128 element probe."""
    return [
        # one plane wave of a 64 element probe onto a small image, the beamformer's default interpolation: live imaging
        dict(name="live_frame", path="das", geo="tabbed", kind="korder_cubic", param=8, sum="tx_and_rx", nfr=0,
             ntx=1, nrx=64, nt=1024, nx=64, nz=128),
        # one compound frame at ordinary sizes, default interpolation, geometry given as points
        dict(name="frame_default", path="das", geo="diverging", kind="korder_cubic", param=8, sum="tx_and_rx", nfr=0,
             ntx=31, nrx=128, nt=2048, nx=256, nz=256),
        # one full compound frame, natural cubic
        dict(name="frame_cubic_full", path="das", geo="plane", kind="cubic", param=1, sum="tx_and_rx", nfr=0,
             ntx=75, nrx=128, nt=4096, nx=512, nz=512),
        # the benchmark's batch: 16 full compound frames, natural cubic
        dict(name="batch16_cubic_full", path="das", geo="plane", kind="cubic", param=1, sum="tx_and_rx", nfr=16,
             ntx=75, nrx=128, nt=4096, nx=512, nz=512),
        # a cine loop with odd sizes over delay tables, default interpolation
        dict(name="cine_odd_default", path="das", geo="tabbed", kind="korder_cubic", param=8, sum="tx_and_rx", nfr=12,
             ntx=11, nrx=127, nt=1999, nx=201, nz=333),
        # delay multiply and sum over the receive channels, linear interpolation
        dict(name="dmas_linear", path="dmas", geo="tabbed", kind="linear", param=1, nfr=0,
             ntx=15, nrx=96, nt=2048, nx=150, nz=400, nlag=10, dmastype="ssr"),
        # short-lag spatial coherence image of one compound frame
        dict(name="slsc_cubic", path="slsc", geo="diverging", kind="cubic", param=1, nfr=0,
             ntx=31, nrx=128, nt=2048, nx=128, nz=1024, precision="fp16"),
        # image and channel-data gradient of the table-driven beamformer at the benchmark's adjoint size
        dict(name="train_tabbed", path="train_tabbed", geo="tabbed", kind="cubic", param=1, nfr=0, grads="rf",
             ntx=31, nrx=128, nt=4096, nx=256, nz=256),
        # channel-data and sound-speed gradients of the point-driven beamformer
        dict(name="train_synthetic", path="train_synthetic", geo="diverging", kind="linear", param=1, nfr=0,
             ntx=16, nrx=64, nt=2048, nx=192, nz=256),
        # one loss and gradient of a sound-speed map fit
        dict(name="sound_speed_step", path="sos", ntx=11, nrx=64, nt=2048, nx=128, nz=128, nzm=32, nxm=32),
        # demodulation of every line of per-receive images (the benchmark's size)
        dict(name="demod_lines", path="demod", rows=32768, n=2048),
        # a ragged batch of image and coherence requests from several probes
        dict(name="ragged_batch", path="batch", nreq=10, side=256, ntx=31, nrx=128, nt=2048, shape=7),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(("das",) * 6 + ("dmas", "slsc", "train_tabbed", "train_synthetic", "sos", "demod", "batch"))
    if path == "demod":
        n = rng.choice((256, 512, 1024, 2048, 4096, rng.randint(200, 3000)))
        return dict(path=path, rows=_log(rng, 64, min(40000, (1 << 26) // n)), n=n)
    if path == "batch":
        return dict(path=path, nreq=rng.randint(2, 16), side=rng.randint(64, 256), ntx=_log(rng, 3, 40),
                    nrx=rng.randint(48, 128), nt=rng.randint(1024, 4096), shape=rng.randint(0, 1000))
    if path == "sos":
        return dict(path=path, ntx=rng.randint(5, 21), nrx=rng.randint(32, 128), nt=rng.randint(1200, 4096),
                    nx=rng.randint(60, 160), nz=rng.randint(60, 160), nzm=rng.randint(8, 64), nxm=rng.randint(8, 64))
    while True:
        c = dict(path=path, geo=rng.choice(("tabbed", "tabbed", "diverging", "plane")),
                 kind=rng.choice(("korder_cubic", "korder_cubic", "cubic", "cubic", "linear", "nearest")), param=1,
                 nfr=0 if rng.random() < 0.5 else _log(rng, 1, 16), ntx=_log(rng, 1, 75), nrx=rng.randint(24, 160),
                 nt=_log(rng, 512, 6000), nx=_log(rng, 40, 512), nz=_log(rng, 64, 1024))
        if path in ("slsc", "train_synthetic"):
            c["geo"] = "diverging"
        if path == "train_tabbed":
            c.update(geo="tabbed", grads=rng.choice(("rf", "rf", "all")))
        if path.startswith("train") and c["kind"] == "nearest":
            c["kind"] = "linear"
        if c["kind"] == "korder_cubic":
            c["param"] = rng.choice((4, 8, 8, 8, 10))
        if c["kind"] == "nearest":
            c["param"] = rng.choice((1, 1, 4))
        if path == "das":
            c["sum"] = rng.choice(("tx_and_rx",) * 5 + ("tx_only", "rx_only", "none"))
        if path == "dmas":
            c.update(nlag=rng.randint(2, 16), dmastype=rng.choice(("ssr", "pssr")))
        if path == "slsc":
            c.update(nrx=rng.randint(64, 160), kind=rng.choice(("cubic", "cubic", "korder_cubic")),
                     precision=rng.choice(("fp16", "fp16", "bf16", "fp32")))
            c["param"] = 8 if c["kind"] == "korder_cubic" else 1
        f = max(1, c["nfr"])
        chan, pix = c["ntx"] * c["nrx"], c["nx"] * c["nz"]
        kept = {"none": chan, "tx_only": c["nrx"], "rx_only": c["ntx"]}.get(c.get("sum"), c["nrx"] if path != "das" else 1)
        most = 3e9 if path in ("das", "dmas", "slsc") else 2.5e8 / (2 if c.get("grads") == "all" else 1)
        if 1e6 < f * chan * pix < most and f * kept * pix < 4e8 and f * chan * c["nt"] < 2e8:
            return c


# ------------------------------------------------------------------ inputs ---
def _rand(seed, *shape):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    return torch.randn(shape, generator=g, device="cuda")


def _channels(seed, frames, ntx, nrx, nt):
    """Channel data like diffuse scattering gives: noise in the probe's band (5 MHz, 60 %), falling with depth."""
    f = torch.fft.rfftfreq(nt, 1.0 / FS, device="cuda")
    band = torch.exp(-0.5 * ((f - FC) / (0.25 * FC)) ** 2)
    fall = torch.exp(-1.5 * torch.arange(nt, device="cuda") / nt)
    rf = torch.empty((frames, ntx, nrx, nt), device="cuda")
    for i in range(frames):
        x = torch.fft.irfft(torch.fft.rfft(_rand(seed * 1009 + i, ntx, nrx, nt)) * band, n=nt)
        rf[i] = x * fall / x.std()
    return rf


def _probe(case):
    """Element positions, steering angles and the x-major pixel grid (float64)."""
    xele = PITCH * (np.arange(case["nrx"]) - (case["nrx"] - 1) / 2)
    steers = np.radians(np.linspace(-16, 16, case["ntx"])) if case["ntx"] > 1 else np.zeros(1)
    half = max(abs(xele[0]), 5e-3)
    x = np.linspace(-half, half, case["nx"])
    z = np.linspace(3e-3, min(45e-3, 0.4 * case["nt"] / FS * C0), case["nz"])
    X, Z = np.meshgrid(x, z, indexing="ij")
    return xele, steers, np.stack([X.ravel(), Z.ravel()], axis=1)


def _tables(case):
    """Plane-wave delay tables and a Hann f/1.5 receive apodisation, float32."""
    xele, steers, pnts = (torch.as_tensor(a, device="cuda") for a in _probe(case))
    x, z = pnts[:, 0][None], pnts[:, 1][None]
    first = torch.where(steers <= 0, xele[-1], xele[0])[:, None]
    tautx = ((x - first) * torch.sin(steers)[:, None] + z * torch.cos(steers)[:, None]) / C0
    dx = x - xele[:, None]
    half = z / (2 * FNUM)
    apodrx = torch.where(dx.abs() <= half, 0.5 * (1 + torch.cos(math.pi * dx / half)), torch.zeros_like(dx))
    taurx = torch.sqrt(dx * dx + z * z) / C0
    return tuple(t.float().contiguous() for t in (tautx, torch.ones_like(tautx), taurx, apodrx))


def _waves(case):
    """The point geometry's arrays (float32): plane waves as points 10 m behind the probe, or diverging waves."""
    xele, steers, pnts = _probe(case)
    n = np.stack([np.sin(steers), np.cos(steers)], axis=1)
    if case["geo"] == "plane":
        first = np.stack([np.where(steers <= 0, xele[-1], xele[0]), 0 * steers], axis=1)
        o = -10.0 * n
        d = first - o
        t0 = np.sum(n * (o - first), axis=1) / C0
        ala = np.arccos(np.abs(np.sum(d * n, axis=1)) / np.linalg.norm(d, axis=1))
    else:
        r = max(1.2 * abs(xele[0]), 8e-3)
        o = -r * n
        t0 = -np.min(np.hypot(o[:, 0, None] - xele, o[:, 1, None]), axis=1) / C0
        ala = np.full(len(steers), 0.75)
    rx = np.stack([xele, 0 * xele], axis=1)
    nrx = len(xele)
    f = dict(ovectx=o, nvectx=n, t0tx=t0, alatx=ala, doftx=0 * t0, ovecrx=rx,
             nvecrx=np.stack([np.zeros(nrx), np.ones(nrx)], axis=1), alarx=np.full(nrx, np.arctan2(0.5, FNUM)), pnts=pnts)
    return {**{k: np.ascontiguousarray(v, dtype=np.float32) for k, v in f.items()}, "c0": C0}


def _interp(case):
    if case["kind"] == "korder_cubic":
        return {"kind": "korder_cubic", "k": case["param"]}
    return {"kind": "nearest", "usf": case["param"]} if case["kind"] == "nearest" else {"kind": case["kind"]}


def _beamformer(case):
    from pycbf_amd import gpu
    from pycbf_amd.gpu import advanced
    tabbed = case["geo"] == "tabbed"
    if tabbed:
        geo = dict(zip(("tautx", "apodtx", "taurx", "apodrx"), _tables(case)))
    else:
        geo = _waves(case)
    geo.update(t0=0.0, dt=1.0 / FS, nt=case["nt"], interp=_interp(case), device="cuda")
    if case["path"] == "dmas":
        cls = advanced.TabbedDMASBeamformer if tabbed else advanced.SyntheticDMASBeamformer
        return cls(**geo, lags=np.arange(1, case["nlag"] + 1), dmastype=case["dmastype"])
    if case["path"] == "slsc":
        return advanced.SyntheticSLSCBeamformer(**geo, lags=np.array(SLSC_LAGS), gridshape=(case["nx"], case["nz"]), kwin=SLSC_KWIN,
                                                dsfz=SLSC_KWIN, precision=case["precision"])
    cls = gpu.TabbedBeamformer if tabbed else gpu.SyntheticBeamformer
    return cls(**geo, sumtype=case.get("sum", "tx_and_rx"))


def _requests(case):
    """The ragged batch's requests: (case of its geometry, kind) each; sizes spread around the case's."""
    r = np.random.default_rng(case["shape"])
    out = []
    for i in range(case["nreq"]):
        side = max(24, int(case["side"] * r.uniform(0.5, 1.4)))
        out.append((dict(geo="diverging", ntx=max(1, int(case["ntx"] * r.uniform(0.2, 1.6))), nrx=max(32, int(case["nrx"] * r.uniform(0.5, 1.5))),
                         nt=case["nt"], nx=side, nz=side, kind="cubic", param=1), "slsc" if i % 4 == 3 else "das"))
    return out


def _cotangent(case, seed):
    shape = (case["nx"] * case["nz"],)
    return _rand(seed + 77, *(((case["nfr"],) if case["nfr"] else ()) + shape))


def _sos_inputs(case, seed):
    xele, steers, pnts = _probe(case)
    x, z = pnts[:, 0], pnts[:, 1]
    box = (float(x[0]), float(z[0]), (x[-1] - x[0]) / case["nxm"], (z[-1] - z[0]) / case["nzm"])
    f = lambda a: torch.as_tensor(np.ascontiguousarray(a, np.float32), device="cuda")  # noqa: E731
    first = np.where(steers <= 0, xele[-1], xele[0])
    cmap = C0 + 15.0 * torch.nn.functional.avg_pool2d(_rand(seed + 5, 1, 1, case["nzm"] + 2, case["nxm"] + 2), 3, 1)[0, 0]
    return dict(rf=_channels(seed, 1, case["ntx"], case["nrx"], case["nt"])[0], steer=f(steers), xorig=f(first), xele=f(xele), pvec=f(pnts)), box, cmap


def prepare(case, seed):
    path = case["path"]
    if path == "demod":
        x = torch.fft.irfft(torch.fft.rfft(_rand(seed, case["rows"], case["n"])) * _line_band(case["n"]), n=case["n"])
        return dict(case=case, rf=x.contiguous())
    if path == "batch":
        from pycbf_amd.gpu.batch import BatchRequest, RaggedBatch
        reqs = _requests(case)
        b = RaggedBatch([BatchRequest(params=_waves(q), gridshape=(q["nx"], q["nz"]), kind=k, lags=SLSC_LAGS, kwin=SLSC_KWIN, dsfz=SLSC_KWIN if k == "slsc" else 1)
                         for q, k in reqs], nt=case["nt"], dt=1.0 / FS)
        for i, (q, _) in enumerate(reqs):
            b.rf_views[i].copy_(_channels(seed * 31 + i, 1, q["ntx"], q["nrx"], q["nt"])[0])
        b.autotune()
        b.capture()
        return dict(case=case, batch=b)
    if path == "sos":
        from pycbf_amd.gpu.sos import SlownessGrid, SoSProblem
        d, box, cmap = _sos_inputs(case, seed)
        prob = SoSProblem(**d, gridshape=(case["nx"], case["nz"]), geo=SlownessGrid(case["nzm"], case["nxm"], *box), t0=0.0, dt=1.0 / FS, c0=C0, smooth_weight=1e-3)
        return dict(case=case, prob=prob, cmap=cmap.requires_grad_())
    rf = _channels(seed, max(1, case["nfr"]), case["ntx"], case["nrx"], case["nt"])
    rf = rf if case["nfr"] else rf[0]
    s = dict(case=case, rf=rf)
    if path == "train_tabbed":
        s["tabs"] = [t.requires_grad_(case["grads"] == "all") for t in _tables(case)]
    else:
        s["bf"] = _beamformer(case)
    if path.startswith("train"):
        s["g"] = _cotangent(case, seed)
        s["rf"] = rf.requires_grad_()
    if path == "train_synthetic":
        s["c0"] = torch.tensor(C0, dtype=torch.float32, requires_grad=True)
    return s


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "demod":
        from pycbf_amd.gpu.demod import fft_tukey_demod
        return fft_tukey_demod(s["rf"], *_band(case["n"]))
    if path == "batch":
        s["batch"].run()
        return list(s["batch"].outputs)
    if path == "sos":
        loss = s["prob"].angle_loss(s["cmap"])
        return [loss.detach(), *torch.autograd.grad(loss, [s["cmap"]])]
    if path == "train_tabbed":
        from pycbf_amd.gpu.autograd import das_tabbed
        k = case["param"] if case["kind"] == "korder_cubic" else None
        out = das_tabbed(s["rf"], *s["tabs"], 0.0, 1.0 / FS, case["kind"], "tx_and_rx", THRESH, k=k)
        return [out.detach(), *torch.autograd.grad(out, [s["rf"]] + (s["tabs"] if case["grads"] == "all" else []), s["g"])]
    if path == "train_synthetic":
        from pycbf_amd.gpu.autograd import das_synthetic
        out = das_synthetic(s["rf"], s["bf"], s["c0"])
        return [out.detach(), *torch.autograd.grad(out, [s["rf"], s["c0"]], s["g"])]
    return s["bf"](s["rf"], out_as_numpy=False)


# -------------------------------------------------------------------- work ---
def work(case):
    """Inputs read once, outputs written once; per (tx, rx, pixel) the delay and weight sums, and on the third of
    them inside an f/1.5 aperture the interpolation of each frame."""
    path = case["path"]
    if path == "demod":
        n, rows = case["n"], case["rows"]
        return {"bytes": rows * (4 * n + 8 * _bins(n)[1]), "flops": rows * 5 * n * math.log2(n)}
    if path == "batch":
        b = f = 0
        for q, kind in _requests(case):
            chan, pix = q["ntx"] * q["nrx"], q["nx"] * q["nz"]
            b += 4 * chan * q["nt"] + 8 * pix + 4 * pix // (SLSC_KWIN if kind == "slsc" else 1)
            f += chan * pix * (2 + 8 / 3)
        return {"bytes": b, "flops": f}
    chan, pix, elem, fr = case["ntx"] * case["nrx"], case["nx"] * case["nz"], case["ntx"] + case["nrx"], max(1, case.get("nfr", 0))
    rf = 4 * fr * chan * case["nt"]
    per = {"nearest": 2, "linear": 4}.get(case.get("kind", "cubic"), 8)
    kept = {"none": chan, "tx_only": case["nrx"], "rx_only": case["ntx"]}.get(case.get("sum"), 1)
    geo = 8 * elem * pix if case.get("geo") == "tabbed" else 8 * pix
    flops = chan * pix * (2 + fr * per / 3)
    if path == "sos":
        return {"bytes": rf + 8 * pix, "flops": 3 * flops + 2 * 64 * 10 * elem * pix}
    if path.startswith("train"):
        more = rf + (geo if case.get("grads") == "all" else 0)
        return {"bytes": rf + geo + 8 * fr * pix + more, "flops": 2 * flops}
    if path == "slsc":
        flops += fr * (pix // SLSC_KWIN) * case["nrx"] / 3 * (4 * SLSC_KWIN + 2 * SLSC_KWIN * len(SLSC_LAGS))
        return {"bytes": rf + geo + 4 * fr * pix // SLSC_KWIN, "flops": flops}
    if path == "dmas":
        flops += fr * pix * case["nrx"] * case["nlag"] * 3
    return {"bytes": rf + geo + 4 * fr * kept * pix, "flops": flops}


# ------------------------------------------------------ the same in 64 bits ---
def _spline(y):
    """dt^2 y'' of the natural cubic spline through y (..., n): (1, 4, 1) z = 6 second differences, odd about both ends."""
    n = y.shape[-1]
    r = torch.nn.functional.pad(6.0 * (y[..., 2:] - 2.0 * y[..., 1:-1] + y[..., :-2]), (1, 1))
    e = torch.cat([r, -r[..., 1:-1].flip(-1)], dim=-1)
    k = torch.arange(e.shape[-1] // 2 + 1, device=y.device, dtype=y.dtype)
    return torch.fft.irfft(torch.fft.rfft(e) / (4.0 + 2.0 * torch.cos(2 * math.pi * k / e.shape[-1])), n=e.shape[-1])[..., :n]


def _slopes(y, k):
    """Slopes at both ends of every interval from the not-a-knot spline through the k samples around it."""
    C = np.diag(np.full(k, 4.0)) + np.diag(np.ones(k - 1), 1) + np.diag(np.ones(k - 1), -1)
    P = 3.0 * (np.diag(np.ones(k - 1), 1) - np.diag(np.ones(k - 1), -1))
    C[0], C[-1], P[0], P[-1] = 0, 0, 0, 0
    C[0, :2], P[0, :3] = (1, 2), (-2.5, 2.0, 0.5)
    C[-1, -2:], P[-1, -3:] = (2, 1), (-0.5, -2.0, 2.5)
    S = torch.as_tensor(np.linalg.solve(C, P), device=y.device)
    n = y.shape[-1]
    j = torch.arange(n - 1, device=y.device)
    w = (j - (k - 1) // 2).clamp(0, n - k)  # first sample of the interval's window
    d = y.unfold(-1, k, 1) @ S.T
    return d[..., w, j - w], d[..., w, j - w + 1]


def _at(y, x, kind, param):
    """Values at the times x (R, P) of the traces y (R, n), zero off the trace."""
    n = y.shape[-1]
    q = x / DT
    if kind == "nearest":
        it = torch.floor(q * param + 0.5)
        on = (it >= 0) & (it <= param * (n - 1))
        it = it.clamp(0, param * (n - 1))
        if param == 1:
            return torch.gather(y, 1, it.long()) * on
        q, kind = it / param, "cubic"
    else:
        on = (q >= 0) & (q <= n - 1)
    j = q.detach().floor().clamp(0, n - 2).long()
    b = q - j
    a = 1.0 - b
    y0, y1 = torch.gather(y, 1, j), torch.gather(y, 1, j + 1)
    if kind == "korder_cubic":
        d0, d1 = (torch.gather(d, 1, j) for d in _slopes(y, param))
        v = y0 + b * (d0 + b * (3 * (y1 - y0) - 2 * d0 - d1 + b * (2 * (y0 - y1) + d0 + d1)))
    else:
        v = a * y0 + b * y1
        if kind == "cubic":
            z = _spline(y)
            v = v + ((a ** 3 - a) * torch.gather(z, 1, j) + (b ** 3 - b) * torch.gather(z, 1, j + 1)) / 6.0
    return v * on


def _geometry(w, scale=1.0):
    """(tautx, apodtx, taurx, apodrx) of the point geometry in 64 bits; `scale` multiplies every path."""
    t = {k: torch.as_tensor(v, device="cuda").double() for k, v in w.items() if k != "c0"}
    d = t["pnts"][None] - t["ovectx"][:, None]
    mag, proj = d.norm(dim=-1), (d * t["nvectx"][:, None]).sum(-1)
    tautx = (torch.sign(proj) * mag / C0 + t["t0tx"][:, None]) * scale
    apodtx = (torch.acos((proj / mag).abs().clamp(max=1.0)) <= t["alatx"][:, None]).double()
    d = t["pnts"][None] - t["ovecrx"][:, None]
    mag, proj = d.norm(dim=-1), (d * t["nvecrx"][:, None]).sum(-1)
    apodrx = (torch.acos((proj / mag).clamp(-1.0, 1.0)) <= t["alarx"][:, None]).double()
    return tautx, apodtx, mag / C0 * scale, apodrx


def _das(rf, tabs, kind, param, sumtype, thresh=THRESH):
    """rf (F, ntx, nrx, nt): the beamformers' output with the frame axis first, in 64 bits."""
    tautx, apodtx, taurx, apodrx = (t.double() for t in tabs)
    frames = []
    for f in range(rf.shape[0]):
        acc, sep = 0.0, []
        for t in range(rf.shape[1]):
            w = apodtx[t][None] * apodrx
            v = _at(rf[f, t].double(), tautx[t][None] + taurx, kind, param) * (w * (w.abs() >= thresh))
            if sumtype in ("tx_and_rx", "tx_only"):
                acc = acc + (v if sumtype == "tx_only" else v.sum(0))
            else:
                sep.append(v if sumtype == "none" else v.sum(0))
        frames.append(torch.stack(sep) if sep else acc)
    return torch.stack(frames)


def _coherence(im, apodrx, nx, nz):
    """Short-lag spatial coherence of per-receive images (nrx, nx nz): windows of SLSC_KWIN samples clipped to the grid,
    elements with a non-zero weight over the whole window (neighbours in a row), correlations averaged over pairs, then lags."""
    K, nrx = SLSC_KWIN, im.shape[0]
    win = lambda v, fill: torch.nn.functional.pad(v.reshape(-1, nx, nz), (K // 2, K), value=fill).unfold(-1, K, K)[..., : -(-nz // K), :]  # noqa: E731
    x, on = win(im, 0.0), win(torch.ones_like(im[:1]), 0.0)
    use = (win((apodrx != 0).double(), 1.0) > 0).all(-1)
    cnt = on.sum(-1, keepdim=True)
    c = (x - x.sum(-1, keepdim=True) / cnt) * on
    sd = torch.sqrt((c * c).sum(-1, keepdim=True) / cnt)
    ok = use & (sd[..., 0] >= 1e-10)
    z = torch.where(ok[..., None], c / (sd * torch.sqrt(cnt)), torch.zeros_like(c))
    out = 0.0
    for m in SLSC_LAGS:
        pair = (ok[:-m] & ok[m:]).sum(0)
        out = out + (z[:-m] * z[m:]).sum(-1).sum(0) / pair
    out = out / len(SLSC_LAGS)
    return torch.where(use.sum(0) > max(SLSC_LAGS), out, torch.zeros_like(out))


def _line_band(n):
    """The lines' spectrum: the band that _band(n) keeps, and some noise around it."""
    lo, m = _bins(n)
    k = torch.arange(n // 2 + 1, device="cuda")
    return 0.02 + torch.exp(-0.5 * ((k - lo - m / 2) / (m / 4)) ** 2)


def _band(n):
    """(kmin, kmax, ks): 5 .. 12 MHz of two-way travel at 19.5 um axial spacing."""
    return 2 * 5e6 / C0, 2 * 12e6 / C0, 1.0 / 19.5e-6


def _bins(n):
    kmin, kmax, ks = _band(n)
    f = np.fft.rfftfreq(n, 1 / ks)
    lo, hi = int(np.argmin(np.abs(f - kmin))), int(np.argmin(np.abs(f - kmax))) + 1
    return lo, hi - lo


def _demod(x):
    lo, m = _bins(x.shape[-1])
    k = np.arange(m)
    edge = int(np.floor(0.25 * (m - 1) / 2.0))  # Tukey window, a quarter of it tapered
    w = np.ones(m)
    w[:edge + 1] = 0.5 * (1 + np.cos(np.pi * (2.0 * k[:edge + 1] / 0.25 / (m - 1) - 1)))
    w[m - edge - 1:] = 0.5 * (1 + np.cos(np.pi * (2.0 * k[m - edge - 1:] / 0.25 / (m - 1) - 2.0 / 0.25 + 1)))
    X = torch.fft.rfft(x.double())[..., lo:lo + m] * torch.as_tensor(w, device=x.device)
    return torch.fft.ifft(torch.roll(X, -(m // 2), dims=-1))


def _rays(slow, box, shape, d, elem):
    """Straight-ray delay to every pixel of element `elem` (transmits first) through the bilinear slowness map, 64 midpoints."""
    nzm, nxm = shape
    p = d["pvec"].double()
    px, pz = p[:, 0], p[:, 1]
    ntx = d["steer"].numel()
    fire = 0.0
    if elem < ntx:
        a = d["steer"][elem].double()
        qx = px - pz * torch.tan(a)
        L = pz / torch.cos(a)
        fire = (qx - d["xorig"][elem].double()) * torch.sin(a) / C0
    else:
        qx = d["xele"][elem - ntx].double().expand_as(px)
        L = torch.sqrt((px - qx) ** 2 + pz ** 2)
    t = ((torch.arange(64, device=px.device, dtype=torch.float64) + 0.5) / 64)[:, None]
    f32 = [float(np.float32(b)) for b in box]
    u = ((qx + t * (px - qx) - f32[0]) / f32[2] - 0.5).clamp(0, nxm - 1)
    v = ((t * pz - f32[1]) / f32[3] - 0.5).clamp(0, nzm - 1)
    k, i = u.floor().clamp(max=nxm - 2).long(), v.floor().clamp(max=nzm - 2).long()
    wx, wz = u - k, v - i
    s = slow.reshape(-1)
    at = i * nxm + k
    top = s[at] + wx * (s[at + 1] - s[at])
    bot = s[at + nxm] + wx * (s[at + nxm + 1] - s[at + nxm])
    return fire + L * (top + wz * (bot - top)).mean(0)


def _sos_exact(case, seed):
    d, box, cmap = _sos_inputs(case, seed)
    c = cmap.double().requires_grad_()
    slow32 = (1.0 / cmap).double()  # the map's slowness as the kernels receive it
    slow = slow32.clone().requires_grad_()
    shape = (case["nzm"], case["nxm"])
    ntx, nrx = case["ntx"], case["nrx"]
    with torch.no_grad():
        tau = torch.stack([_rays(slow, box, shape, d, e) for e in range(ntx + nrx)])
    tau.requires_grad_()
    one = torch.ones_like(tau[:1])
    im = torch.cat([torch.stack([_das(d["rf"][None, t:t + 1], (tau[t:t + 1], one, tau[ntx:], one.expand(nrx, -1)), "cubic", 1, "tx_and_rx", 0.0)[0]])
                    for t in range(ntx)])
    diff = im[3:] - im[:-3]
    rough = ((c[1:] - c[:-1]) ** 2).mean() + ((c[:, 1:] - c[:, :-1]) ** 2).mean()
    loss = (diff * diff).sum() / (im * im).sum() + 1e-3 * rough
    gtau, gc = torch.autograd.grad(loss, [tau, c])
    for e in range(ntx + nrx):
        g = torch.autograd.grad(_rays(slow, box, shape, d, e), [slow], gtau[e])[0]
        gc = gc - g * slow32 * slow32
    return [loss.detach(), gc]


def _train_exact(case, seed):
    rf = _channels(seed, max(1, case["nfr"]), case["ntx"], case["nrx"], case["nt"])
    g = _cotangent(case, seed).double().reshape(rf.shape[0], -1)
    scale = torch.ones((), dtype=torch.float64, device="cuda", requires_grad=True)
    tabbed = case["path"] == "train_tabbed"
    tabs = [t.double().detach() for t in (_tables(case) if tabbed else _geometry(_waves(case)))]
    every = tabbed and case["grads"] == "all"
    out, grf, gtab, gscale = 0.0, [], [torch.zeros_like(t) for t in tabs], 0.0
    for t in range(case["ntx"]):  # the image is a sum over transmits: one transmit's graph at a time
        x = rf[:, t:t + 1].double().requires_grad_()
        use = [tabs[0][t:t + 1], tabs[1][t:t + 1], tabs[2], tabs[3]]
        use = [u.clone().requires_grad_(every) for u in use]
        o = _das(x, (use[0] * scale, use[1], use[2] * scale, use[3]), case["kind"], case["param"], "tx_and_rx")
        got = torch.autograd.grad(o, [x, scale] + (use if every else []), g)
        out = out + o.detach()
        grf.append(got[0].float())
        gscale = gscale + got[1]
        for k, q in enumerate(got[2:]):
            if k < 2:
                gtab[k][t] = q[0]
            else:
                gtab[k] += q
    grf = torch.cat(grf, dim=1).double()
    if not case["nfr"]:
        out, grf = out[0], grf[0]
    if tabbed:
        return [out, grf] + (gtab if every else [])
    return [out, grf, -gscale / C0]  # every delay is a path over c0


def exact(case, seed):
    path = case["path"]
    if path == "demod":
        return _demod(prepare(case, seed)["rf"])
    if path == "sos":
        return _sos_exact(case, seed)
    if path.startswith("train"):
        return _train_exact(case, seed)
    if path == "batch":
        outs = []
        for i, (q, kind) in enumerate(_requests(case)):
            tabs = _geometry(_waves(q))
            rf = _channels(seed * 31 + i, 1, q["ntx"], q["nrx"], q["nt"])
            im = _das(rf, tabs, "cubic", 1, "tx_only" if kind == "slsc" else "tx_and_rx")[0]
            outs.append(_coherence(im, tabs[3], q["nx"], q["nz"]) if kind == "slsc" else im.reshape(q["nx"], q["nz"]))
        return outs
    rf = _channels(seed, max(1, case["nfr"]), case["ntx"], case["nrx"], case["nt"])
    tabs = _tables(case) if case["geo"] == "tabbed" else _geometry(_waves(case))
    sumtype = case["sum"] if path == "das" else "tx_only"
    im = _das(rf, tabs, case["kind"], case["param"], sumtype)
    if path == "slsc":
        im = torch.stack([_coherence(f, tabs[3], case["nx"], case["nz"]) for f in im])
    if path == "dmas":
        per = [f[:-m] * f[m:] for f in im for m in range(1, case["nlag"] + 1)]
        if case["dmastype"] == "ssr":
            per = [(torch.sign(q) * torch.sqrt(q.abs())).sum(0) for q in per]
        else:
            per = [q.sum(0) for q in per]
        im = torch.stack(per).reshape(im.shape[0], case["nlag"], -1).sum(1)
        if case["dmastype"] == "pssr":
            im = torch.sign(im) * torch.sqrt(im.abs())
    return im if case["nfr"] else im[0]
