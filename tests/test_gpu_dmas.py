"""GPU DMAS against the FP64 restatement of the notebook formulas."""
import numpy as np
import pytest

import oracle
from oracle import numerics
from pycbf_amd.gpu import SyntheticDMASBeamformer, TabbedDMASBeamformer
from tests.helpers import assert_close_to_peak, small_synthetic, small_tabbed

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def small():
    return small_tabbed(nrx=24)


@pytest.mark.parametrize("dmastype", ["ssr", "power", "pssr"])
@pytest.mark.parametrize("sumlags", [True, False])
@pytest.mark.parametrize("lagaxis", ["rx", "tx"])
def test_tabbed_dmas(small, dmastype, sumlags, lagaxis):
    tautx, apodtx, taurx, apodrx = small["tabs"]
    lags = np.array([1, 2, 3, 5]) if lagaxis == "rx" else np.array([1, 2])
    bf = TabbedDMASBeamformer(tautx=tautx, taurx=taurx, apodtx=apodtx, apodrx=apodrx,
                              t0=small["t0"], dt=small["dt"], nt=small["nt"],
                              interp={"kind": "cubic"}, lags=lags, lagaxis=lagaxis,
                              dmastype=dmastype, sumlags=sumlags)
    got = bf(small["rf"])
    sumtype = "tx_only" if lagaxis == "rx" else "rx_only"
    imsep = oracle.das_tabbed(small["rf"], small["t0"], small["dt"], *small["tabs"],
                              kind="cubic", sumtype=sumtype)
    ref = numerics.dmas(imsep, lags, dmastype, sumlags)
    assert got.shape == ref.shape
    assert_close_to_peak(got, ref, 1e-4, f"{dmastype} sumlags={sumlags} axis={lagaxis}")


def test_dmas_lag_values_are_used(small):
    """Lag 3 alone differs from lag 1 alone (the reference used 0..nlag-1)."""
    tautx, apodtx, taurx, apodrx = small["tabs"]
    outs = []
    for lags in ([1], [3]):
        bf = TabbedDMASBeamformer(tautx=tautx, taurx=taurx, apodtx=apodtx, apodrx=apodrx,
                                  t0=small["t0"], dt=small["dt"], nt=small["nt"],
                                  interp={"kind": "linear"}, lags=np.array(lags),
                                  dmastype="power")
        outs.append(bf(small["rf"]))
    assert not np.allclose(outs[0], outs[1])


def test_synthetic_dmas_frames():
    w = small_synthetic(ntx=4, nrx=16)
    p = w["params"]
    rfs = np.stack([w["rf"], 2.0 * w["rf"]])
    bf = SyntheticDMASBeamformer(**p, t0=w["t0"], dt=w["dt"], nt=w["nt"],
                                 interp={"kind": "cubic"}, lags=np.arange(1, 4),
                                 dmastype="power")
    got = bf(rfs)
    for f in range(2):
        imsep = oracle.das_synthetic(rfs[f], w["t0"], w["dt"], p["ovectx"], p["nvectx"],
                                     p["t0tx"], p["alatx"], p["doftx"], p["ovecrx"], p["nvecrx"],
                                     p["alarx"], p["c0"], p["pnts"], kind="cubic",
                                     sumtype="tx_only")
        ref = numerics.dmas(imsep, np.arange(1, 4), "power", True)
        assert_close_to_peak(got[f], ref, 1e-4, f"frame {f}")


def _dmas(im, lags, dmastype, sumlags):
    import torch
    from pycbf_amd.gpu import _engine as E
    nfr, nsep, npx = im.shape
    d = torch.as_tensor(im, device="cuda")
    L = torch.as_tensor(np.asarray(lags, np.int32), device="cuda")
    out = torch.empty((nfr, npx) if sumlags else (nfr, len(lags), npx), dtype=torch.float32, device="cuda")
    E.check(E.lib.pycbf_dmas(E.ptr(d), nfr, nsep, npx, E.ptr(L), len(lags), E.DMASTYPE[dmastype], int(sumlags),
                             E.ptr(out), E.stream_of(d.device)), "pycbf_dmas")
    return out.cpu().numpy()


@pytest.mark.parametrize("nsep,npx,nfr", [(1, 1, 1), (7, 63, 2), (8, 64, 1), (9, 65, 3), (41, 130, 1), (252, 70, 1),
                                          (253, 70, 1)])
def test_dmas_columns_and_lags_at_their_edges(nsep, npx, nfr):
    """Blocks of eight elements with remainders, columns of 252 elements (the
    tallest held in LDS) and 253, lags that pair nothing.  Bar: 1e-5 of the
    peak (float32 sums against FP64)."""
    im = np.random.default_rng(nsep).standard_normal((nfr, nsep, npx)).astype(np.float32)
    lags = [1, 0, 3, -2, nsep - 1, nsep, nsep + 5]
    for dmastype in ("ssr", "power", "pssr"):
        for sumlags in (True, False):
            got = _dmas(im, lags, dmastype, sumlags)
            for f in range(nfr):
                assert_close_to_peak(got[f], numerics.dmas(im[f], lags, dmastype, sumlags), 1e-5,
                                     f"{nsep} {dmastype} {sumlags}")


@pytest.mark.parametrize("nsep,npx,nfr", [(2, 40, 1), (3, 16384, 2), (3, 32767, 1), (6, 65537, 2), (6, 131071, 1),
                                          (9, 57344, 4), (10, 70000, 4)])
def test_dmas_of_short_columns(nsep, npx, nfr):
    """Columns of few elements on both sides of the pixel count from which each
    lane walks its own; lags apart leave the columns at another height.  Bar as
    above, for the P-DMAS-SSR on the sums under its root: among so many pixels some
    sums are near zero, where the root of a rounding error is far above it."""
    im = np.random.default_rng(nsep).standard_normal((nfr, nsep, npx)).astype(np.float32)
    lags = list(range(1, nsep))
    for dmastype in ("ssr", "power", "pssr"):
        for sumlags in (True, False):
            got = _dmas(im, lags, dmastype, sumlags)
            under = (lambda x: np.sign(x) * np.asarray(x, np.float64) ** 2) if dmastype == "pssr" else np.asarray
            for f in range(nfr):
                assert_close_to_peak(under(got[f]), under(numerics.dmas(im[f], lags, dmastype, sumlags)), 1e-5,
                                     f"{nsep} {dmastype} {sumlags}")


def test_dmas_of_infinities_and_nans():
    """Infinite, NaN and zero elements count as in the column-free kernel, which
    the same columns padded with zeros to 300 elements take."""
    rng = np.random.default_rng(1)
    im = rng.standard_normal((1, 30, 200)).astype(np.float32)
    for v in (np.inf, -np.inf, np.nan, 0.0):
        im[0][rng.random((30, 200)) < 0.03] = v
    tall = np.concatenate([im, np.zeros((1, 270, 200), np.float32)], axis=1)
    for sumlags in (True, False):
        got, ref = (_dmas(x, [1, 2, 5], "ssr", sumlags) for x in (im, tall))
        assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
        fin = np.isfinite(ref)
        assert np.array_equal(np.sign(got[~fin & ~np.isnan(ref)]), np.sign(ref[~fin & ~np.isnan(ref)]))
        assert_close_to_peak(got[fin], ref[fin], 1e-5, "finite outputs")
