"""Bucketing of particles into deposit tiles at the sizes where its split of
the work changes: workgroups of one and of several chunks, tile counts within
and beyond the counters' LDS window, catalogues in space order and shuffled
(pairs inside and outside the window), positions on cell and half-cell
boundaries (where the shifted grid's cells follow the FP64 expression), part
tables passed as kernel arguments and copied.  A tile's sums are integers at a
scale set by its record count, so any order of a catalogue gives the same
bits; the FP64 oracle says whether they are the right ones."""
import numpy as np
import pytest

from tests.test_gpu_parity import _check

pytestmark = pytest.mark.gpu

L = 640.0


def _catalogue(n, Ng, seed, lattice):
    rng = np.random.default_rng(seed)
    d = np.empty((n, 4))
    if lattice:   # multiples of half a cell, a few a rounding away from them
        x = rng.integers(0, 2 * Ng, (n, 3)) * (0.5 * L / Ng)
        d[:, :3] = np.clip(x + rng.choice([0.0, 0.0, 1e-13, -1e-13], (n, 3)), 0,
                           np.nextafter(L, 0))
    else:
        d[:, :3] = rng.uniform(0.0, L, (n, 3))
    d[:, 3] = rng.uniform(0.5, 1.5, n)
    return d[np.lexsort((d[:, 2], d[:, 1], d[:, 0]))]


@pytest.mark.parametrize("scheme", [0, 1, 2, 3])
@pytest.mark.parametrize("Ng,tile,n,lattice", [
    (32, (8, 8, 8), 1, False),
    (32, (8, 8, 8), 255, True),
    (64, (8, 16, 64), 131073, False),      # one particle past 256 per workgroup
    (48, (4, 4, 16), 30011, True),
    (256, (4, 4, 4), 40009, False),        # 262144 tiles: windows
    (256, (4, 8, 8), 300007, True),        # 65536 tiles: windows
])
def test_order_and_oracle(psh, oracle, scheme, Ng, tile, n, lattice):
    d = _catalogue(n, Ng, 100 + n, lattice)
    kw = dict(gsize=Ng, assign=scheme, intlace=True, bsize=L, kbin=0.02, poles=[0, 2, 4])
    ctx = psh.Context(psh.make_conf(**kw))
    ctx.set_tiles(tile)
    w = float(d[:, 3].sum())
    got = []
    for order in (np.arange(n), np.random.default_rng(1).permutation(n), np.arange(n)[::-1]):
        dev = psh.DeviceArray.from_numpy(np.ascontiguousarray(d[order]))
        got.append(ctx.run_device(dev, n, w))
    for g in got[1:]:
        assert np.array_equal(g["pl"][0], got[0]["pl"][0])
    if n > 1:
        ref = oracle.run(oracle.make_conf(**kw), [d])
        _check(got[0], ref, [0, 2, 4], ref["shot"][0])


@pytest.mark.parametrize("nmock", [8, 9])   # the last table passed as arguments, the first copied
def test_batch_parts(psh, nmock):
    kw = dict(gsize=64, assign=psh.TSC, intlace=True, bsize=L, kbin=0.02, poles=[0, 2])
    cats = [_catalogue(1 + 900 * m * m, 64, m, m % 2 == 1) for m in range(nmock)]
    off = np.concatenate([[0], np.cumsum([len(c) for c in cats])])
    dev = psh.DeviceArray.from_numpy(np.concatenate(cats))
    ws = [float(c[:, 3].sum()) for c in cats]
    ctx = psh.Context(psh.make_conf(**kw), nmock_max=nmock)
    for graph in (False, True, True):
        got = ctx.run_batch(dev, off, ws, graph=graph)
        for c, w, g in zip(cats, ws, got):
            one = psh.Context(psh.make_conf(**kw)).run_device(
                psh.DeviceArray.from_numpy(c), len(c), w)
            # the weight scale of a launch is its largest weight, so a mock's
            # integers may sit at another power of two than alone
            s = np.abs(one["pl"][0][0]) + L ** 3 / w
            assert np.all(np.abs(g["pl"][0] - one["pl"][0]) <= 1e-5 * s)


def test_record_overflow_reruns(psh, oracle):
    """Every particle at a corner of eight tiles: more records than the buffer
    expects, found when the run's results arrive; the run is repeated with a
    larger buffer, and the next one fits at once."""
    Ng, n = 64, 30000
    rng = np.random.default_rng(3)
    d = np.empty((n, 4))
    d[:, :3] = (8 * rng.integers(0, Ng // 8, (n, 3)) + 7.6) * (L / Ng)
    d[:, 3] = 1.0
    kw = dict(gsize=Ng, assign=psh.PCS, intlace=True, bsize=L, kbin=0.02, poles=[0, 2, 4])
    ref = oracle.run(oracle.make_conf(**kw), [d])
    dev = psh.DeviceArray.from_numpy(d)
    for graph in (None, False, True):
        ctx = psh.Context(psh.make_conf(**kw))
        ctx.set_tiles((8, 8, 8))
        for _ in range(2):
            got = (ctx.run_device(dev, n, float(n)) if graph is None else
                   ctx.run_batch(dev, [0, n], [float(n)], graph=graph)[0])
            _check(got, ref, [0, 2, 4], ref["shot"][0])


@pytest.mark.parametrize("scheme,tile,n", [
    (2, (32, 32, 32), 50000),    # rows of whole quads would not fit the LDS
    (1, (8, 16, 32), 600000),    # many records per thread, aligned rows
    (0, (4, 4, 64), 60000),      # one tile spans z, odd row offset
    (3, (64, 4, 4), 60000),      # one tile spans x
])
@pytest.mark.parametrize("order", ["sorted", "shuffled"])
def test_deposit_tiles(psh, oracle, scheme, tile, n, order):
    d = _catalogue(n, 64, 7, False)
    if order == "shuffled":
        d = d[np.random.default_rng(2).permutation(n)]
    kw = dict(gsize=64, assign=scheme, intlace=False, bsize=L, kbin=0.02, poles=[0, 2, 4])
    ctx = psh.Context(psh.make_conf(**kw))
    ctx.set_tiles(tile)
    got = ctx.run_device(psh.DeviceArray.from_numpy(d), n, float(d[:, 3].sum()))
    ref = oracle.run(oracle.make_conf(**kw), [d])
    _check(got, ref, [0, 2, 4], ref["shot"][0])
