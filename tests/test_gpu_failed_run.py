"""A run that fails leaves what the last good run left: the |mu| cells and the
feature rows made from them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_alias_rows_after_a_failed_run(psh):
    L, n = 1000.0, 200000
    rng = np.random.default_rng(4)
    d = np.empty((n, 4))
    d[:, :3] = rng.uniform(0.0, L, (n, 3))
    d[:, 3] = 1.0
    conf = psh.make_conf(gsize=64, assign=psh.CIC, bsize=L, kbin=0.02, poles=[0, 2, 4])
    ctx = psh.Context(conf)
    ctx.set_mu_cells(8)
    ctx.run_device(psh.DeviceArray.from_numpy(d), n, float(n))
    cells, rows = ctx.cells(), ctx.alias_rows()
    bad = d[:1000].copy()
    bad[10, 1] = L                         # outside [0, BOX_SIZE)
    with pytest.raises(psh.PshError) as e:
        ctx.run_device(psh.DeviceArray.from_numpy(bad), len(bad), 500.0)
    assert e.value.code == psh.ERR_CATA
    assert np.array_equal(ctx.cells(), cells)
    assert np.array_equal(ctx.alias_rows(), rows)
