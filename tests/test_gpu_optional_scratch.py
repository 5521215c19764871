"""Scratch that a run can do without gives way to what it needs: the bucket
ranges of the count pass (kept for meshes of any tile count) when there is no
memory for them and the record buffer."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = 640.0


def _uniform(n, seed):
    rng = np.random.default_rng(seed)
    d = np.empty((n, 4))
    d[:, :3] = rng.uniform(0.0, L, (n, 3))
    d[:, 3] = rng.uniform(0.5, 1.5, n)
    return d


@pytest.fixture
def faults(psh):
    yield psh
    psh.fault_inject(psh.FAULT_ALLOC, 0)


@pytest.mark.parametrize("graph", [None, False, True])
@pytest.mark.parametrize("k", [1, 2])
def test_one_allocation_less_for_a_larger_run(faults, k, graph):
    """A context that ran a small catalogue (262144 tiles, enough particles
    for the ranges) grows its buffers for a larger one; any one of the two
    allocations may fail."""
    P = faults
    m0, n = 530000, 1200000
    small, large = _uniform(m0, 1), _uniform(n, 2)
    w = float(large[:, 3].sum())
    conf = P.make_conf(gsize=256, assign=P.TSC, intlace=True, bsize=L, kbin=0.02)
    ds, dl = P.DeviceArray.from_numpy(small), P.DeviceArray.from_numpy(large)
    ctx = P.Context(conf)
    ctx.set_tiles((4, 4, 4))

    def run(dev, m, ws):
        if graph is None:
            return ctx.run_device(dev, m, ws)
        return ctx.run_batch(dev, [0, m], [ws], graph=graph)[0]

    run(ds, m0, float(small[:, 3].sum()))
    P.fault_inject(P.FAULT_ALLOC, k)
    first = run(dl, n, w)
    P.fault_inject(P.FAULT_ALLOC, 0)
    ref = P.Context(conf)
    ref.set_tiles((4, 4, 4))
    want = ref.run_device(dl, n, w)
    for got in (first, run(dl, n, w)):
        assert np.array_equal(got["cnt"], want["cnt"])
        assert np.array_equal(got["pl"][0], want["pl"][0])
