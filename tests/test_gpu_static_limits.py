"""psh_run_device_static at the end of its scratch: catalogue sizes that once
filled it to the last 256 bytes still fit, and a particle outside the box is
reported as that where the scratch has 57344 bytes left for the coordinate
bounds of the message."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = 1000.0


def _run(psh, dev, n, **kw):
    conf = psh.make_conf(bsize=L, poles=[0, 2, 4], **kw)
    return psh.run_device_static(conf, dev, n, float(n), psh.Context(conf).nbin())


# the largest catalogues that the scratch took with log bins when they had no
# table of live tiles (found by bisection on an MI355X)
FULL = [(16, False, 1, 5851497), (64, True, 1, 5052411), (128, True, 3, 3417477)]


@pytest.fixture(scope="module")
def catalogue():
    n = max(f[3] for f in FULL)
    d = np.empty((n, 4))
    d[:, :3] = np.random.default_rng(1).uniform(0, L, (n, 3))
    d[:, 3] = 1.0
    return d


@pytest.mark.parametrize("Ng,intlace,scheme,n", FULL)
def test_log_bins_fill_the_scratch(psh, catalogue, Ng, intlace, scheme, n):
    kw = dict(gsize=Ng, assign=scheme, intlace=intlace, logscale=True, kmin=-2.2, kbin=0.05)
    dev = psh.DeviceArray.from_numpy(catalogue)
    res = _run(psh, dev, n, **kw)
    assert res["cnt"].sum() > 0


def test_box_error_with_little_scratch_left(psh, catalogue):
    Ng, intlace, scheme, full = FULL[1]
    n = full - 1500                                 # 53 bytes each: about 80 KB left
    d = catalogue[:n].copy()
    d[n // 2, 0] = L
    dev = psh.DeviceArray.from_numpy(d)
    with pytest.raises(psh.PshError) as e:
        _run(psh, dev, n, gsize=Ng, assign=scheme, intlace=intlace, logscale=True, kmin=-2.2,
             kbin=0.05)
    assert e.value.code == psh.ERR_CATA
    assert "not smaller than BOX_SIZE" in str(e.value)
