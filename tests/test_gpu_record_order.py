"""The order in which the PCS deposit, and the TSC deposit into tiles of whole
z rows, takes a bucket's records: a stretch of consecutive records per thread,
where the bucket holds more than one per thread and is in space order; whole
waves where it is not."""
import numpy as np
import pytest

from tests.test_gpu_parity import _check

pytestmark = pytest.mark.gpu


# one tile of 4096 cells, 256 threads: stretches of equal length, one or
# several whole waves with one record more, part of a wave with one more
@pytest.mark.parametrize("n", [256, 257, 319, 320, 512, 513, 767, 768, 1000, 4113])
@pytest.mark.parametrize("order", ["sorted", "shuffled"])
def test_every_record_once(psh, oracle, n, order):
    L = 160.0
    rng = np.random.default_rng(n)
    d = np.empty((n, 4))
    d[:, :3] = rng.uniform(0.0, L, (n, 3))
    d[:, 3] = rng.uniform(0.5, 1.5, n)
    if order == "sorted":
        d = d[np.lexsort((d[:, 2], d[:, 1], d[:, 0]))]
    kw = dict(gsize=16, assign=psh.PCS, intlace=True, bsize=L, kbin=0.05, poles=[0, 2, 4])
    ctx = psh.Context(psh.make_conf(**kw))
    ctx.set_tiles((16, 16, 16))
    got = ctx.run_device(psh.DeviceArray.from_numpy(d), n, float(d[:, 3].sum()))
    ref = oracle.run(oracle.make_conf(**kw), [d])
    _check(got, ref, [0, 2, 4], ref["shot"][0])


# tiles of whole z rows have 1024 threads
@pytest.mark.parametrize("n", [16384, 16385, 60000])
@pytest.mark.parametrize("scheme", [2, 3])
def test_whole_z_rows(psh, oracle, n, scheme):
    L = 128.0
    rng = np.random.default_rng(n)
    d = np.empty((n, 4))
    d[:, :3] = rng.uniform(0.0, L, (n, 3))
    d[: n // 2, 0] = 4.5 * d[: n // 2, 0] / L + 0.2      # half of them in few tiles
    d[: n // 2, 1] = 4.5 * d[: n // 2, 1] / L + 0.2
    d[:, 3] = rng.uniform(0.5, 1.5, n)
    d = d[np.lexsort((d[:, 2], d[:, 1], d[:, 0]))]
    kw = dict(gsize=128, assign=scheme, intlace=True, bsize=L, kbin=0.1, poles=[0, 2, 4])
    ctx = psh.Context(psh.make_conf(**kw))
    ctx.set_tiles(psh.fused_tile(128, True))
    got = ctx.run_device(psh.DeviceArray.from_numpy(d), n, float(d[:, 3].sum()))
    ref = oracle.run(oracle.make_conf(**kw), [d])
    _check(got, ref, [0, 2, 4], ref["shot"][0])


@pytest.mark.parametrize("scheme,fused", [(3, False), (2, True)])
def test_dense_ordered_catalogue_is_not_slower(psh, scheme, fused):
    """Space order, in which neighbouring records meet in one cell, against
    the same catalogue shuffled: with neighbours side by side in a wave the
    deposit of four particles per cell takes 1.6 times as long (TSC in whole
    z rows 1.4 times)."""
    d, n = psh.gen_clustered_box(ng=256, L=1000.0, f=0.8, seed=5, npart=8e6)
    h = d.to_numpy((n, 4))
    s = psh.DeviceArray.from_numpy(h[np.random.default_rng(1).permutation(n)])
    ms = []
    for dev in (d, s):
        ctx = psh.Context(psh.make_conf(gsize=128, assign=scheme, intlace=True, bsize=1000.0,
                                        kbin=0.01))
        if fused:
            ctx.set_tiles(psh.fused_tile(128, True))
        ctx.set_profiling(True)
        t = []
        for _ in range(8):
            ctx.run_device(dev, n, float(n))
            t.append(ctx.timings()[4])
        ms.append(float(np.median(t[2:])))
    assert ms[0] < (1.15 if fused else 1.3) * ms[1], ms
