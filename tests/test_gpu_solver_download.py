"""Solver.download beside the solver's other uses: from a thread whose current device is another one, and while
another thread runs the solver."""
import ctypes
import threading

import numpy as np
import pytest

import slamplay_amd as S

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
