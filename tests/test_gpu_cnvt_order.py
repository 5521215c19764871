"""Order search of the coordinate conversion on the device: the order of the
host's search for any redshift range, over one and several arrays (bounds
folded array by array, empty ones skipped), and its error cases."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _sky(n, zlo, zhi, seed):
    rng = np.random.default_rng(seed)
    d = np.column_stack([rng.uniform(0, 360, n), rng.uniform(-90, 90, n),
                         rng.uniform(zlo, zhi, n), np.ones(n)])
    if n:
        d[0, 2] = zlo
        d[-1, 2] = zhi
    return d


@pytest.mark.parametrize("ol,w", [(None, -1.0), (0.6, -1.0), (None, -0.8), (0.75, -1.1)])
@pytest.mark.parametrize("sizes,zlo,zhi,err", [
    ((1,), 0.5, 0.5, 1e-8), ((255,), 0.0, 0.1, 1e-6), ((257, 0, 1), 0.4, 0.7, 1e-8),
    ((70000, 300000), 0.01, 6.0, 1e-12), ((1000, 3, 0, 5), 0.0, 20.0, 1e-9)])
def test_order_and_distances(psh, ol, w, sizes, zlo, zhi, err):
    cv = psh.make_cnvt(omega_m=0.31, omega_l=ol, eos_w=w, ecdst=err)
    cats = [_sky(n, zlo + 0.1 * i * (zhi - zlo) / 8, zhi, 3 + i) for i, n in enumerate(sizes)]
    dev = [psh.DeviceArray.from_numpy(c if len(c) else np.zeros((1, 4))) for c in cats]
    z = np.concatenate([c[:, 2] for c in cats])
    ref = O.cmvdist_order(cv.omega_m, cv.omega_l, cv.omega_k, O.eos_widx(w), err, z.min(), z.max())
    assert ref > 0
    assert psh.cnvt_device(cv, [(d, len(c)) for d, c in zip(dev, cats)]) == ref
    for d, c in zip(dev, cats):
        if len(c):
            want = O.cnvt(c, om=cv.omega_m, ol=cv.omega_l, ok=cv.omega_k, eos_w=w, order=ref)
            # up to 33 positive terms of a few ulp each, both sides: 25 ulp
            r = np.linalg.norm(want[:, :3], axis=1)
            assert np.all(np.abs(d.to_numpy((len(c), 4))[:, :3] - want[:, :3]) <= 1e-14 * r[:, None])


@pytest.mark.parametrize("w", [-1.0, -0.9])
@pytest.mark.parametrize("zmin,err", [(-1e-9, 1e-8), (0.1, -1.0)])   # negative z; never converges
def test_errors_leave_records(psh, w, zmin, err):
    cat = _sky(5000, 0.1, 0.9, 1)
    cat[17, 2] = zmin
    dev = psh.DeviceArray.from_numpy(cat)
    with pytest.raises(psh.PshError) as e:
        psh.cnvt_device(psh.make_cnvt(eos_w=w, ecdst=err), [(dev, len(cat))])
    assert e.value.code == psh.ERR_CNVT
    assert np.array_equal(dev.to_numpy((len(cat), 4)), cat)
    assert psh.cnvt_device(psh.make_cnvt(eos_w=w), [(dev, 0)]) == 0
