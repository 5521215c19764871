"""Boxes in units that take the grid's numbers to the ends of their range:
sides so large that FP32 |k|^2 is denormal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("logscale", [False, True])
@pytest.mark.parametrize("poles,los", [([0, 2, 4], [0, 0, 1]), ([0, 1, 2], [1, 0, 0])])
def test_denormal_wave_numbers(psh, logscale, poles, los):
    """Lengths times 2^57 (a box side of 1.4e20): every FP64 step scales
    exactly, FP32 |k|^2 of the lowest modes is denormal with 20 bits left,
    so mu^2 there is off by up to 2^-20 and P_l by (2l + 1) l (l + 1) / 2 of
    that."""
    s = 2.0 ** 57
    L, n, Ng = 1000.0, 30000, 32
    rng = np.random.default_rng(6)
    c = rng.uniform(0, L, (40, 3))
    d = np.empty((n, 4))
    d[:, :3] = (c[rng.integers(0, 40, n)] + rng.normal(0, 30.0, (n, 3))) % L
    d[:, 3] = 1.0
    res = []
    for f in (1.0, s):
        kw = dict(gsize=Ng, assign=psh.CIC, intlace=True, bsize=L * f, poles=poles, los=los)
        if logscale:
            kw.update(logscale=True, kmin=np.log10(0.005 / f), kbin=0.2)
        else:
            kw.update(kbin=0.01 / f)
        e = d.copy()
        e[:, :3] *= f
        res.append(psh.Context(psh.make_conf(**kw)).run_device(
            psh.DeviceArray.from_numpy(e), n, float(n)))
    a, b = res
    assert np.array_equal(a["cnt"], b["cnt"])
    scale = np.abs(a["pl"][0][0]) + L ** 3 / n
    for li, ell in enumerate(poles):
        tol = 1e-6 + (2 * ell + 1) * ell * (ell + 1) / 2 * 2.0 ** -20
        assert np.all(np.abs(b["pl"][0][li] / s ** 3 - a["pl"][0][li]) <= tol * scale), ell
