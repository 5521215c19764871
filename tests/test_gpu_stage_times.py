"""Stage times (psh_ctx_timings) where a run is more than one chain of
launches: a batch that fills only part of its context's meshes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = 1000.0


def _uniform(n, seed):
    rng = np.random.default_rng(seed)
    d = np.empty((n, 4))
    d[:, :3] = rng.uniform(0.0, L, (n, 3))
    d[:, 3] = 1.0
    return d


def test_zy_split_of_a_partial_batch(psh):
    """The y passes' share of the z and y time does not depend on whether the
    two grids' meshes are adjacent: with one mock less than the context
    holds they are not.  (y alone of the second grid, against z and y of the
    first and z of the second, would be a quarter instead of a half.)"""
    nmax, n = 5, 20000
    conf = psh.make_conf(gsize=256, assign=psh.CIC, intlace=True, bsize=L, kbin=0.02)
    dev = psh.DeviceArray.from_numpy(_uniform(nmax * n, 1))
    ctx = psh.Context(conf, nmock_max=nmax)
    ctx.set_profiling(True)
    share = {}
    for nm in (nmax, nmax - 1):
        reps = []
        for _ in range(9):
            ctx.run_batch(dev, [n * m for m in range(nm + 1)], [float(n)] * nm)
            ms = ctx.timings()
            assert ms[5] > 0 and ms[6] > 0
            reps.append(ms[6] / (ms[5] + ms[6]))
        share[nm] = float(np.median(reps))
    assert abs(share[nmax] - share[nmax - 1]) < 0.12, share
