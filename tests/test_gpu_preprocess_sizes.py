"""Device Normalize and Perturb where their kernels divide the work: blocks of the selection, generator
workgroups and chunks, one value on every point, both signs and a wide range of magnitudes."""
import time

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


def _degenerate(kind, n):
    """Maps on which most keys of a selection share their first bits."""
    rng = np.random.default_rng(n)
    p = rng.normal(0.0, 3.0, (n, 3))
    if kind == "plane":
        p[:, 2] = 5.0
    elif kind == "most on a plane":
        p[rng.random(n) < 0.6, 1] = 5.0
    elif kind == "thin plane":  # 60% within 1e-9 of it, some on either side
        flat = rng.random(n) < 0.6
        p[flat, 0] = 5.0 + 1e-9 * p[flat, 0]
    elif kind == "far from the origin":
        p += np.array([5e5, 4.2e6, -1e3])
    elif kind == "one point":
        p[:] = [1.5, -2.5, 3.5]
        p[0] += 1.0  # (the largest distance; the median is zero, and so the scale infinite, without any)
    elif kind == "two values":
        p = rng.choice([-1.5, 2.25], (n, 3))
    return p


def _one_camera(pts):
    n = len(pts)
    cams = np.array([0.1, -0.2, 0.05, 0.3, -0.1, -5.0, 500.0, 0.0, 0.0])
    return cams, S.BALProblem.from_arrays(np.zeros(n, np.int32), np.arange(n, dtype=np.int32), np.zeros((n, 2)), cams,
                                          pts.reshape(-1))


# 2^17 points: the largest number whose last bits one block finds from all keys alike; beyond it more
# histograms take part, and the block has at most 2^14 keys
@pytest.mark.parametrize("kind", ["plain", "plane", "most on a plane", "thin plane", "far from the origin", "one point",
                                  "two values"])
@pytest.mark.parametrize("n", [1, 3, 1025, 8193, 131072, 131073, 300001])
def test_device_normalize_degenerate_maps(oracle_mod, kind, n):
    pts = _degenerate(kind, n)
    cams, p = _one_camera(pts)
    sv = S.Solver(p)
    sv.normalize()
    gc, got = sv.download()
    sv.close()
    rc, ref = oracle_mod.normalize(1, n, cams, pts.reshape(-1))
    # medians are elements of the input and the transform rounds as the oracle's: equal bits (a scale of 100 / 0
    # included)
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("n", [100000, 400000])
def test_device_normalize_of_degenerate_maps_takes_no_multiple(n):
    def median_us(kind):
        _, p = _one_camera(_degenerate(kind, n))
        sv = S.Solver(p)
        t = []
        for _ in range(15):
            sv.reset()
            start = time.perf_counter()
            sv.normalize()
            t.append(time.perf_counter() - start)
        sv.close()
        return 1e6 * float(np.median(t))

    plain = median_us("plain")
    for kind in ("plane", "far from the origin", "one point"):
        # up to two and a half times for the passes over all keys that only such maps need; with all of their
        # keys left to one block of the plain maps' size it was 7 to 45 times
        assert median_us(kind) < 4 * plain, (kind, plain)
