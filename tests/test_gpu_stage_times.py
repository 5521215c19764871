"""Stage times (psh_ctx_timings) where a run is more than one chain of
launches: a batch that fills only part of its context's meshes, and a run
repeated after its records overflowed their buffer."""
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


def test_assignment_time_after_an_overflow(psh):
    """Particles at corners of eight tiles overflow the record buffer once;
    the assignment time of the run that is reported holds none of the first
    run's transforms."""
    Ng, n = 512, 100000
    rng = np.random.default_rng(2)
    d = np.empty((n, 4))
    d[:, :3] = (8 * rng.integers(0, Ng // 8, (n, 3)) + 7.6) * (L / Ng)
    d[:, 3] = 1.0
    conf = psh.make_conf(gsize=Ng, assign=psh.PCS, intlace=True, bsize=L, kbin=0.02)
    ctx = psh.Context(conf)
    ctx.set_tiles((8, 8, 8))
    ctx.set_profiling(True)
    few = psh.DeviceArray.from_numpy(_uniform(100, 3))
    for _ in range(2):
        ctx.run_device(few, 100, 100.0)
    ctx.run_device(psh.DeviceArray.from_numpy(d), n, float(n))
    ms = ctx.timings()
    # [0] less the bucketing and deposit kernels: what came before them
    assert ms[0] - ms[4] - ms[7] < 0.5 * (ms[1] + ms[2]), ms
