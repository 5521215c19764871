"""Deposit of both grids in more workgroups than one launch may have threads
for (2^32): at N_g = 1024 4x4x8 tiles, 8388608 per grid, with 256 threads each,
4x4x4 tiles with 128.  The tile shape sets the fixed-point step of the cells
only, so the spectra agree with the default tiles' to that step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [(4, 4, 8), (4, 4, 4)])
def test_interlaced_small_tiles_1024(psh, tile):
    L, n = 1000.0, 50000
    rng = np.random.default_rng(5)
    d = np.empty((n, 4))
    d[:, :3] = rng.uniform(0.0, L, (n, 3))
    d[:, 3] = rng.uniform(0.5, 1.5, n)
    w = float(d[:, 3].sum())
    dev = psh.DeviceArray.from_numpy(d)
    ctx = psh.Context(psh.make_conf(gsize=1024, assign=psh.CIC, intlace=True, bsize=L, kbin=0.05))
    want = ctx.run_device(dev, n, w)
    ctx.set_tiles(tile)
    assert ctx.tiles() == tile
    got = ctx.run_device(dev, n, w)
    assert np.array_equal(got["cnt"], want["cnt"])
    scale = np.abs(want["pl"][0][0]) + L ** 3 / w
    assert np.all(np.abs(got["pl"][0] - want["pl"][0]) <= 1e-5 * scale)
