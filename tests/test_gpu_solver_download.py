"""Solver.download beside the solver's other uses: from a thread whose current device is another one, and while
another thread runs the solver."""
import ctypes
import threading

import numpy as np
import pytest

import slamplay_amd as S
from slamplay_amd import _capi as C

pytestmark = pytest.mark.gpu

FIXED = dict(max_num_iterations=4, function_tolerance=0.0, gradient_tolerance=0.0, parameter_tolerance=0.0)


def test_download_with_another_current_device():
    if S.device_count() < 2:
        pytest.skip("needs two devices")
    p = S.synthetic(2, seed=3, num_cameras=6, num_points=200, max_track=6)
    start = p.cameras().copy(), p.points().copy()
    sv = S.Solver(p, device=1, **FIXED)
    hip = ctypes.CDLL("libamdhip64.so")
    assert hip.hipSetDevice(0) == 0
    got = sv.download()
    sv.close()
    np.testing.assert_array_equal(got[0], start[0])
    np.testing.assert_array_equal(got[1], start[1])


# each iteration's kernels launched one by one (launch_mode 1), so that a download's kernel can run between any two
@pytest.mark.parametrize("solver", ["dense", "pcg"])
def test_downloads_beside_a_run_do_not_change_it(solver):
    kw = dict(FIXED, launch_mode=1, linear_solver=C.SOLVER_DENSE_SCHUR if solver == "dense" else C.SOLVER_ITERATIVE_SCHUR)
    p = S.synthetic(2, seed=5, num_cameras=24, num_points=3000, max_track=10)
    sv = S.Solver(p, **kw)
    alone = sv.run()["final_cost"]
    ref = sv.download()
    stop = threading.Event()
    reads = [0]

    def read():
        while not stop.is_set():
            sv.download()
            reads[0] += 1

    t = threading.Thread(target=read)
    t.start()
    try:
        for _ in range(20):
            sv.reset()
            # every sum runs in a fixed order: the same bits
            assert sv.run()["final_cost"] == alone
            for got, want in zip(sv.download(), ref):
                np.testing.assert_array_equal(got, want)
    finally:
        stop.set()
        t.join()
    sv.close()
    assert reads[0] > 0
