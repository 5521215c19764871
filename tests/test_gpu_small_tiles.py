"""Deposit tiles of less than 2048 cells, 128 threads each where there are
8192 workgroups or more: buckets at the edges of their threads and of several
rounds of them, rows of 4 to 16 cells, 32- and 64-bit cells; and the time of
very many of them."""
import numpy as np
import pytest

from tests.test_gpu_parity import _check, _survey_cats

pytestmark = pytest.mark.gpu

L = 160.0


def _catalogue(n):
    rng = np.random.default_rng(n)
    d = np.empty((n, 4))
    d[:, :3] = rng.uniform(0.0, L, (n, 3))
    d[:, 3] = rng.uniform(0.5, 1.5, n)
    return d[np.lexsort((d[:, 2], d[:, 1], d[:, 0]))]


# 4096 tiles of 64 cells, 8192 workgroups; one of them with n records more
@pytest.mark.parametrize("scheme", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [126, 127, 128, 129, 255, 256, 257, 1000])
def test_full_tile(psh, oracle, scheme, n):
    d = _catalogue(3000)
    e = _catalogue(n)
    e[:, :3] = 16 * 2.5 + 0.5 + 1.5 * e[:, :3] / L      # inside one cell
    d = np.concatenate([d, e])
    kw = dict(gsize=64, assign=scheme, intlace=True, bsize=L, kbin=0.05, poles=[0, 2])
    ctx = psh.Context(psh.make_conf(**kw))
    ctx.set_tiles((4, 4, 4))
    got = ctx.run_device(psh.DeviceArray.from_numpy(d), len(d), float(d[:, 3].sum()))
    ref = oracle.run(oracle.make_conf(**kw), [d])
    _check(got, ref, [0, 2], ref["shot"][0])


@pytest.mark.parametrize("tile", [(4, 4, 4), (4, 8, 8), (8, 4, 16), (8, 8, 16)])
@pytest.mark.parametrize("Ng", [64, 160])    # fewer than 8192 workgroups and more
def test_shapes(psh, oracle, Ng, tile):
    n = 40000
    d = _catalogue(n)
    kw = dict(gsize=Ng, assign=3, intlace=True, bsize=L, kbin=0.1, poles=[0, 2])
    ctx = psh.Context(psh.make_conf(**kw))
    ctx.set_tiles(tile)
    assert ctx.tiles() == tile
    got = ctx.run_device(psh.DeviceArray.from_numpy(d), n, float(d[:, 3].sum()))
    ref = oracle.run(oracle.make_conf(**kw), [d])
    _check(got, ref, [0, 2], ref["shot"][0])


def test_survey_cells(psh, oracle):
    (dp, dwc, dfkp, dnz), (rp, rwc, rfkp, rnz) = _survey_cats(60000, 5)
    wd, wr, sums = oracle.survey_sums(dwc, dfkp, dnz, rwc, rfkp, rnz)
    d, r = np.column_stack([dp, wd]), np.column_stack([rp, wr])
    kw = dict(gsize=64, assign=2, intlace=True, issim=False, kbin=0.01, poles=[0, 2])
    ctx = psh.Context(psh.make_conf(**kw))
    ctx.set_tiles((4, 4, 4))
    got = ctx.run_host([d], [r], [sums])
    ref = oracle.run(oracle.make_conf(**kw), [d], [r], [sums])
    _check(got, ref, [0, 2], sums["shot"], sums["norm"])


def test_many_tiles_take_no_longer_than_before(psh):
    """262144 tiles of 64 cells, both grids: 0.24 ms with 256 threads for
    both grids of a tile, 0.43 with 256 for each, 0.24 with 128."""
    n = 20000
    dev = psh.DeviceArray.from_numpy(_catalogue(n))
    ctx = psh.Context(psh.make_conf(gsize=256, assign=psh.CIC, intlace=True, bsize=L, kbin=0.05))
    ctx.set_tiles((4, 4, 4))
    ctx.set_profiling(True)
    t = []
    for _ in range(12):
        ctx.run_device(dev, n, float(n))
        t.append(ctx.timings()[4])
    assert np.median(t[2:]) < 0.33, t
