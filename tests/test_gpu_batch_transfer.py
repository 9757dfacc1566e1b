"""Batch results read one window at a time (the first download after a change fetches its window alone,
later ones a packed copy of all): every order of reading gives the parameters the batch holds now."""
import time
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import slamplay_amd as S

pytestmark = pytest.mark.gpu

FIXED = dict(max_num_iterations=3, function_tolerance=0.0, gradient_tolerance=0.0, parameter_tolerance=0.0)


# windows of (cameras, points): a single one, a few (one of them beyond the batched kernels, 36
# cameras, and one of 64 points, one chunk exactly), and enough for two lanes
@pytest.mark.parametrize("sizes", [[(5, 30)], [(5, 65), (36, 200), (8, 64), (6, 200)], [(5 + i % 3, 40 + i) for i in range(66)]])
def test_batch_downloads_follow_the_parameters(sizes):
    probs = [S.synthetic(4, seed=i + 1, num_cameras=c, num_points=n, max_track=min(c, 6)) for i, (c, n) in enumerate(sizes)]
    start = [(p.cameras().copy(), p.points().copy()) for p in probs]
    n = len(probs)

    def alone(w, run):
        """Window w read as the only download after the change."""
        b.reset()
        if run:
            b.run()
        return b.download(w)

    def same(x, y):
        np.testing.assert_array_equal(x[0], y[0])
        np.testing.assert_array_equal(x[1], y[1])

    b = S.Batch(probs, **FIXED)
    some = sorted({0, n // 2, n - 1})
    solved = {w: alone(w, True) for w in some}
    b.reset()
    for w in range(n):
        same(b.download(w), start[w])  # the second one fetches all
    b.run()
    for w in reversed(range(n)):
        got = b.download(w)
        if w in solved:
            same(got, solved[w])
    b.reset()
    for w in some:
        same(b.download(w), start[w])  # not the fetched solution
    b.close()


# windows of the batched kernels beside one of the single-problem solver (36 cameras)
def test_batch_downloads_from_several_threads():
    probs = [S.synthetic(4, seed=i + 1, num_cameras=c, num_points=60 + i, max_track=min(c, 6))
             for i, c in enumerate([5, 36, 8, 6, 7, 5, 36, 9])]
    start = [(p.cameras().copy(), p.points().copy()) for p in probs]
    b = S.Batch(probs, **FIXED)
    b.run()
    b.reset()
    with ThreadPoolExecutor(4) as pool:
        got = list(pool.map(b.download, range(len(probs))))
    for x, y in zip(got, start):
        np.testing.assert_array_equal(x[0], y[0])
        np.testing.assert_array_equal(x[1], y[1])
    b.close()


def _orders(n):
    rng = np.random.default_rng(n)
    yield "up", list(range(n))
    yield "down", list(range(n))[::-1]
    yield "every third", list(range(0, n, 3))
    yield "a few, then up", [n - 1, 0, n // 2] + list(range(n))
    yield "random", list(rng.permutation(n))
    yield "random, repeated", list(rng.integers(0, n, 3 * n))
    yield "one again and again", [n // 3] * (n + 4)
    yield "down from the middle, then up", list(range(n // 2, -1, -1)) + list(range(n))


# how many windows come with a read depends on what was read before (from the third read on, eight for each
# read so far; all, once the reads of one window have cost as much)
@pytest.mark.parametrize("n", [1, 2, 3, 20, 45, 130])
def test_batch_downloads_in_any_order(n):
    # every eighth window is solved by the single-problem solver (36 cameras)
    probs = [S.synthetic(4, seed=i + 1, num_cameras=36 if i % 8 == 5 else 5 + i % 3, num_points=40 + i % 70, max_track=5)
             for i in range(n)]
    b = S.Batch(probs, **FIXED)
    b.run()
    ref = [b.download(w) for w in range(n)]
    for name, order in _orders(n):
        b.reset()
        b.run()
        for w in order:
            got = b.download(w)
            np.testing.assert_array_equal(got[0], ref[w][0], err_msg=f"{name}: window {w}")
            np.testing.assert_array_equal(got[1], ref[w][1], err_msg=f"{name}: window {w}")
    b.close()


def test_reading_two_windows_does_not_fetch_all():
    b = S.Batch(S.local_ba_windows(256, seed=2), max_num_iterations=1)

    def median_ms(windows):
        t = []
        for _ in range(15):
            b.reset()
            start = time.perf_counter()
            for w in windows:
                b.download(w)
            t.append(time.perf_counter() - start)
        return 1e3 * float(np.median(t))

    one, two = median_ms([3]), median_ms([3, 200])
    b.close()
    # two reads of one window each are twice one; all 256 would be more than ten times
    assert two < 5 * one, (one, two)


def test_info_counts_the_packed_copy():
    b = S.Batch([S.synthetic(4, seed=i + 1, num_cameras=5, num_points=40, max_track=5) for i in range(4)], **FIXED)
    before = b.info()["device_bytes"]
    for w in range(4):
        b.download(w)
    values = 4 * (9 * 5 + 3 * 40)
    assert b.info()["device_bytes"] >= before + 8 * values
    b.close()


def test_windows_staged_in_several_groups():
    """One lane's inputs beyond the 64 MB that are staged at a time (2.5 MB a window: 33,000 observations and their
    pairs), a small window among them: every window is where and what it is in a batch of its own."""
    probs = [S.synthetic(4, seed=i + 1, num_cameras=20, num_points=3000, max_track=20) for i in range(44)]
    probs[25] = S.synthetic(4, seed=99, num_cameras=5, num_points=40, max_track=5)
    start = [(p.cameras().copy(), p.points().copy()) for p in probs]
    b = S.Batch(probs, **FIXED)
    assert b.schedule()["lanes"] == 1
    for w in range(len(probs)):
        np.testing.assert_array_equal(b.download(w)[0], start[w][0])
        np.testing.assert_array_equal(b.download(w)[1], start[w][1])
    b.run()
    for w in (0, 24, 25, 26, 43):
        one = S.Batch(probs[w:w + 1], **FIXED)
        one.run()
        np.testing.assert_array_equal(b.download(w)[0], one.download(0)[0])
        np.testing.assert_array_equal(b.download(w)[1], one.download(0)[1])
        one.close()
    b.close()
