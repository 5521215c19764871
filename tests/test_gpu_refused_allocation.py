"""An allocation that the device refuses is reported by its call alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = 640.0


def test_refused_allocation_leaves_no_error(psh):
    """A context too large for the device is refused, and the next run of
    another context is not told of it by its launch checks."""
    n = 20000
    d = np.empty((n, 4))
    d[:, :3] = np.random.default_rng(3).uniform(0.0, L, (n, 3))
    d[:, 3] = 1.0
    dev = psh.DeviceArray.from_numpy(d)
    conf = psh.make_conf(gsize=64, assign=psh.CIC, intlace=True, bsize=L, kbin=0.02)
    ctx = psh.Context(conf)
    want = ctx.run_device(dev, n, float(n))
    with pytest.raises(psh.PshError) as e:        # 32 mocks of 2 x 34.9 GB
        psh.Context(psh.make_conf(gsize=2048, assign=psh.CIC, intlace=True, bsize=L, kbin=0.02),
                    nmock_max=32)
    assert e.value.code == psh.ERR_MEMORY
    got = ctx.run_device(dev, n, float(n))
    assert np.array_equal(got["pl"][0], want["pl"][0])
