"""Device Normalize and Perturb where their kernels divide the work: blocks of the selection, generator
workgroups and chunks, one value on every point, both signs and a wide range of magnitudes."""
import numpy as np
import pytest

import slamplay_amd as S

pytestmark = pytest.mark.gpu


def _points(kind, n):
    rng = np.random.default_rng(n)
    if kind == "two-values":  # the collected keys are half of all points or more
        return rng.choice([-1.5, 2.25], (n, 3))
    if kind == "wide":  # magnitudes over 60 decades, both signs: every digit of the key takes part
        return rng.choice([-1.0, 1.0], (n, 3)) * 10.0 ** rng.uniform(-30, 30, (n, 3))
    return rng.normal(0.0, 3.0, (n, 3)) + np.array([0.0, 1e3, -7.0])


@pytest.mark.parametrize("kind", ["plain", "two-values", "wide"])
@pytest.mark.parametrize("n", [2, 255, 257, 2047, 2049, 33001])
def test_device_normalize_and_perturb_sizes(oracle_mod, kind, n):
    pts = _points(kind, n)
    cams = np.array([0.1, -0.2, 0.05, 0.3, -0.1, -5.0, 500.0, 0.0, 0.0])
    p = S.BALProblem.from_arrays(np.zeros(n, np.int32), np.arange(n, dtype=np.int32), np.zeros((n, 2)), cams, pts.reshape(-1))
    sv = S.Solver(p)
    sv.normalize()
    _, got = sv.download()
    _, ref = oracle_mod.normalize(1, n, cams, pts.reshape(-1))
    # medians are elements of the input and the transform rounds as the oracle's: equal bits
    np.testing.assert_array_equal(got, ref)
    sv.reset()
    sv.perturb(0.1, 0.5, 0.5, seed=n)
    gc, got = sv.download()
    sv.close()
    rc, ref = oracle_mod.perturb(1, n, cams, pts.reshape(-1), 0.1, 0.5, 0.5, seed=n)
    # normals equal to the last ulp of log(); |normal| < 7, sigma 0.5
    np.testing.assert_allclose(got, ref, rtol=1e-15, atol=8 * np.finfo(np.float64).eps)
    np.testing.assert_allclose(gc, rc, rtol=0, atol=1e-12 * np.abs(rc).max())
