"""Binning of the fused x pass: bins decided in FP32 with an error margin and,
within it, by the FP64 expressions, for linear and logarithmic bins whose edges
many modes lie on exactly; the forms of the pole weights (poles 0, 2, 4
with a line of sight without an x component; any others) against the FP64
oracle and against each other."""
import math

import numpy as np
import pytest

from tests.test_gpu_parity import _check, _uniform

pytestmark = pytest.mark.gpu

L = 2.0 * math.pi / 0.01     # fundamental mode 0.01: bin edges on modes


@pytest.mark.parametrize("Ng", [16, 48, 64, 256])
@pytest.mark.parametrize("intlace", [False, True])
@pytest.mark.parametrize("bins", [dict(kbin=0.01), dict(kbin=0.0025, kmax=0.6),
                                  dict(logscale=True, kmin=-2.0, kbin=0.05),
                                  dict(logscale=True, kmin=-1.7, kbin=math.log10(2.0))])
def test_bins_on_edges(psh, oracle, Ng, intlace, bins):
    """A mode in the wrong bin changes it by about 1 / (its modes).  The mesh
    allows 1e-3: a tile's 32-bit cells step by 2^-30 n max(w), each of the
    27 n contributions errs by 0.29 of it, a mode's amplitude is sqrt(n) times
    a window of at least 0.26: 8e-6 in power for n = 500, times 2 l + 1 = 9,
    times 5 standard deviations, and about as much from FP32."""
    n = 500
    d = _uniform(n, [L] * 3, Ng, weights=True)
    kw = dict(gsize=Ng, assign=2, intlace=intlace, bsize=L, poles=[0, 2, 4], **bins)
    if "kmax" in kw and kw["kmax"] > 0.01 * Ng / 2:
        del kw["kmax"]
    got = psh.Context(psh.make_conf(**kw)).run_device(psh.DeviceArray.from_numpy(d), n,
                                                      d[:, 3].sum())
    ref = oracle.run(oracle.make_conf(**kw), [d])
    _check(got, ref, [0, 2, 4], ref["shot"][0], tol=1e-3)


@pytest.mark.parametrize("Ng,intlace", [(32, False), (96, True), (256, True)])
@pytest.mark.parametrize("los", [[0.0, 0.0, 1.0], [0.0, 0.6, 0.8]])
@pytest.mark.parametrize("nmu", [0, 5])
def test_pole_forms_agree(psh, Ng, intlace, los, nmu):
    """Both forms weight the same FP32 |F|^2 and mu: they differ by the rounding
    of the Legendre polynomials, below 4 ulp (5e-7) of a mode's power; P_0's
    weights are exact, so it only differs by the order of FP64 additions."""
    n = 20000
    d = _uniform(n, [L] * 3, 7 + Ng, weights=True)
    dev = psh.DeviceArray.from_numpy(d)
    got = []
    for poles in ([0, 2, 4], [0, 1, 2, 3, 4]):
        ctx = psh.Context(psh.make_conf(gsize=Ng, assign=2, intlace=intlace, bsize=L, kbin=0.02,
                                        poles=poles, los=los))
        if nmu and not intlace:
            ctx.set_mu_cells(nmu)
        got.append(ctx.run_device(dev, n, d[:, 3].sum()))
    fast, gen = got
    assert np.array_equal(fast["cnt"], gen["cnt"])
    shot = L ** 3 / n
    scale = np.abs(gen["pl"][0][0]) + 2 * shot
    for slot, l in enumerate((0, 2, 4)):
        tol = 1e-12 if l == 0 else 5e-7 * (2 * l + 1)
        assert np.all(np.abs(fast["pl"][0][slot] - gen["pl"][0][l]) <= tol * scale), l


@pytest.mark.parametrize("Ng,intlace", [(16, True), (48, False), (256, True)])
@pytest.mark.parametrize("los", [[0.0, 0.0, 1.0], [1.0, 0.0, 0.0], [0.6, 0.0, 0.8]])
def test_pole_sets_agree(psh, Ng, intlace, los):
    """Poles up to 4 directly, in any subset and order; with pole 6 among them
    all by the loop over coefficients.  The same products: the same sums."""
    n = 3000
    d = _uniform(n, [L] * 3, 21 + Ng, weights=True)
    dev = psh.DeviceArray.from_numpy(d)

    def run(poles):
        ctx = psh.Context(psh.make_conf(gsize=Ng, assign=2, intlace=intlace, bsize=L, kbin=0.02,
                                        poles=poles, los=los))
        return dict(zip(poles, ctx.run_device(dev, n, d[:, 3].sum())["pl"][0]))

    ref = run([0, 1, 2, 3, 4, 6])
    scale = np.abs(ref[0]) + 2 * L ** 3 / n
    for poles in ([0], [2], [0, 2], [1, 3], [0, 1, 2, 3, 4]):
        for l, p in run(poles).items():
            assert np.all(np.abs(p - ref[l]) <= 1e-12 * scale), (poles, l)


@pytest.mark.parametrize("Ng", [64, 96])
@pytest.mark.parametrize("kmax", [-0.7, -0.5])
def test_log_bins_below_nyquist(psh, oracle, Ng, kmax):
    """Log bins that end before the Nyquist mode: the passes leave out the tiles
    past the last edge."""
    n = 500
    d = _uniform(n, [L] * 3, Ng, weights=True)
    kw = dict(gsize=Ng, assign=2, intlace=True, bsize=L, poles=[0, 2, 4], logscale=True, kmin=-2.0,
              kmax=kmax, kbin=0.1)
    got = psh.Context(psh.make_conf(**kw)).run_device(psh.DeviceArray.from_numpy(d), n,
                                                      d[:, 3].sum())
    ref = oracle.run(oracle.make_conf(**kw), [d])
    _check(got, ref, [0, 2, 4], ref["shot"][0], tol=1e-3)   # as test_bins_on_edges
