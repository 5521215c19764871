"""Extreme catalogues: coordinates so far from the origin that a cell's
position is no longer exact, and a single particle."""
import numpy as np
import pytest

from tests.test_gpu_parity import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [0, 2])
def test_survey_far_from_origin(psh, oracle, scheme):
    """A survey 2^38 box units away on half-cell positions: the coordinates
    themselves are multiples of 3e-6 cells, so which cell of the shifted grid
    a particle falls into follows the rounding of the reference's expression
    and not the plain grid's fraction (schemes whose window jumps there)."""
    Ng, L, o = 48, 1000.0, 2.0 ** 38
    rng = np.random.default_rng(8)

    def cat(n):
        p = rng.integers(1, 2 * Ng, (n, 3)) * (0.5 * L / Ng) + o
        return np.column_stack([p, rng.uniform(0.5, 1.5, n)])

    d, r = cat(4000), cat(30000)
    alpha = d[:, 3].sum() / r[:, 3].sum()
    sums = dict(wdata=float(d[:, 3].sum()), wrand=float(r[:, 3].sum()), alpha=float(alpha),
                shot=1.2, norm=1e-6)
    kw = dict(gsize=Ng, assign=scheme, intlace=True, issim=False, bsize=L, kbin=0.01, poles=[0])
    got = psh.Context(psh.make_conf(**kw)).run_host([d], [r], [sums])
    ref = oracle.run(oracle.make_conf(**kw), [d], [r], [sums])
    _check(got, ref, [0], sums["shot"], sums["norm"])


@pytest.mark.parametrize("scheme", [0, 1, 2, 3])
def test_one_particle(psh, oracle, scheme):
    """One particle, whose raw power (P plus shot noise) is the alias-corrected
    window's: every mode's |F| is at least (2 / pi)^(scheme + 1), off by at
    most 1e-6 in the FP32 mesh and transforms; twice that relative to |F| in
    the power, 2l + 1 times in a pole."""
    L = 640.0
    kw = dict(gsize=32, assign=scheme, intlace=True, bsize=L, kbin=0.02, poles=[0, 2, 4])
    d = np.array([[123.4, 20.0 * 7.5, 639.99, 1.25]])
    got = psh.Context(psh.make_conf(**kw)).run_device(psh.DeviceArray.from_numpy(d), 1, 1.25)
    ref = oracle.run(oracle.make_conf(**kw), [d])
    assert np.array_equal(got["cnt"], ref["cnt"])
    shot = ref["shot"][0]
    for li, ell in enumerate((0, 2, 4)):
        tol = (2 * ell + 1) * 2e-6 * (np.pi / 2) ** (scheme + 1)
        assert np.all(np.abs(got["pl"][0][li] - ref["pl"][0][li]) <= tol * shot), ell
