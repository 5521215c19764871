"""Bucketing into more than 32768 tiles on both sides of the particle number
from which a workgroup counts in an LDS window of them: global atomics for
every pair below, windows from there on (in the static scratch, which keeps
no ranges, the fill counts again)."""
import numpy as np
import pytest

from tests.test_gpu_parity import _check

pytestmark = pytest.mark.gpu

L = 640.0


def _catalogue(n, seed, order):
    rng = np.random.default_rng(seed)
    d = np.empty((n, 4))
    d[:, :3] = rng.uniform(0.0, L, (n, 3))
    d[:, 3] = rng.uniform(0.5, 1.5, n)
    return d[np.lexsort((d[:, 2], d[:, 1], d[:, 0]))] if order == "sorted" else d


@pytest.mark.parametrize("order", ["sorted", "shuffled"])
@pytest.mark.parametrize("scheme,intlace", [(1, False), (3, True)])
@pytest.mark.parametrize("n", [1, 2 ** 19 - 1, 2 ** 19, 2 ** 19 + 16385])
def test_both_sides(psh, oracle, n, scheme, intlace, order):
    Ng = 160                                   # 64000 tiles
    d = _catalogue(n, n, order)
    w = float(d[:, 3].sum())
    kw = dict(gsize=Ng, assign=scheme, intlace=intlace, bsize=L, kbin=0.02, poles=[0, 2])
    ctx = psh.Context(psh.make_conf(**kw))
    ctx.set_tiles((4, 4, 4))
    got = ctx.run_device(psh.DeviceArray.from_numpy(d), n, w)
    ref = oracle.run(oracle.make_conf(**kw), [d])
    if n > 1:
        _check(got, ref, [0, 2], ref["shot"][0])
    else:   # P + shot noise of one particle: (2l + 1) 2e-6 / |F|, |F| >= (2 / pi)^(scheme + 1)
        for li, ell in enumerate((0, 2)):
            tol = (2 * ell + 1) * 2e-6 * (np.pi / 2) ** (scheme + 1) * ref["shot"][0]
            assert np.all(np.abs(got["pl"][0][li] - ref["pl"][0][li]) <= tol)


@pytest.mark.parametrize("n", [30000, 2 ** 19 + 5])
def test_static_scratch(psh, monkeypatch, n):
    d = _catalogue(n, 9, "sorted")
    w = float(d[:, 3].sum())
    dev = psh.DeviceArray.from_numpy(d)
    conf = psh.make_conf(gsize=160, assign=2, intlace=True, bsize=L, kbin=0.02, poles=[0, 2])
    monkeypatch.setenv("PSH_TILE", "4,4,4")
    ctx = psh.Context(conf)
    assert ctx.tiles() == (4, 4, 4)
    want = ctx.run_device(dev, n, w)
    got = psh.run_device_static(conf, dev, n, w, ctx.nbin())
    assert np.array_equal(got["cnt"], want["cnt"])
    assert np.array_equal(got["pl"][0], want["pl"][0])


def test_few_particles_take_no_longer_than_their_number(psh):
    """20000 particles into 262144 tiles: with windows, three workgroups of
    16384 counters each took 0.20 ms, global atomics take 0.04."""
    n = 20000
    dev = psh.DeviceArray.from_numpy(_catalogue(n, 3, "shuffled"))
    ctx = psh.Context(psh.make_conf(gsize=256, assign=psh.CIC, intlace=True, bsize=L, kbin=0.02))
    ctx.set_tiles((4, 4, 4))
    ctx.set_profiling(True)
    t = []
    for _ in range(12):
        ctx.run_device(dev, n, float(n))
        t.append(ctx.timings()[7])
    assert np.median(t[2:]) < 0.1, t
