"""The dense reduced system at the sizes where its kernels change path: one tile of 32 unknowns, exact
tile multiples, one tile past a 512-row block of the triangular solves and of its second block."""
import numpy as np
import pytest

import slamplay_amd as S
from slamplay_amd import _capi as C

pytestmark = pytest.mark.gpu

FIXED = dict(max_num_iterations=3, function_tolerance=0.0, gradient_tolerance=0.0, parameter_tolerance=0.0)


# 9 nc unknowns: 27 (1 tile), 36, 63 (2 tiles), 180, 189, 198 (6 and 7 tiles), 288 (9 exact), 297,
# 513 (17 tiles: block 2 of one tile), 1026 (33 tiles: block 3 of one tile)
@pytest.mark.parametrize("nc", [3, 4, 7, 20, 21, 22, 32, 33, 57, 114])
def test_dense_sizes_match_oracle(oracle_mod, nc):
    p = S.synthetic(2, seed=nc, num_cameras=nc, num_points=40 * nc, max_track=min(8, nc))
    ref = oracle_mod.solve(p.num_cameras(), p.num_points(), p.camera_index(), p.point_index(), p.observations(),
                           p.cameras(), p.points(), oracle_mod.default_options(**FIXED))
    out = S.SolveBA(p, linear_solver=C.SOLVER_DENSE_SCHUR, **FIXED)
    assert out["num_successful_steps"] == sum(t["step_is_successful"] for t in ref["trace"][1:])
    # both sides solve the same damped FP64 systems: condition number (at most 1e7 in three steps from
    # radius 1e4) times unit roundoff, per step
    assert abs(out["final_cost"] - ref["final_cost"]) <= 1e-8 * ref["final_cost"]
    np.testing.assert_allclose(p.cameras(), ref["cams"], rtol=0, atol=1e-7 * np.abs(ref["cams"]).max())


# Pair lists of the reduced system: observations in random order, points seen twice by one camera (its own
# block then has pairs of two observations), cameras without observations and pairs of cameras without a
# common point (two separate halves).
@pytest.mark.parametrize("nc,repeats", [(5, 0), (6, 1), (13, 7), (66, 40)])
def test_dense_pair_lists_match_oracle(oracle_mod, nc, repeats):
    rng = np.random.default_rng(nc)
    half = S.synthetic(2, seed=nc, num_cameras=nc, num_points=30 * nc, max_track=min(6, nc))
    ci, pi = half.camera_index(), half.point_index()
    no, npt = ci.size, half.num_points()
    obs = half.observations().reshape(-1, 2)
    twice = rng.choice(no, repeats, replace=False)
    order = rng.permutation(2 * no + repeats)
    # the second half's cameras follow an unused one (index nc), its points follow the first half's
    ci = np.concatenate([ci, ci + nc + 1, ci[twice]])[order]
    pi = np.concatenate([pi, pi + npt, pi[twice]])[order]
    ob = np.concatenate([obs, obs, obs[twice] + rng.normal(0, 0.3, (repeats, 2))])[order]
    cams = half.cameras().reshape(-1, 9)
    cams = np.concatenate([cams, cams[:1], cams])
    pts = np.concatenate([half.points(), half.points()])
    p = S.BALProblem.from_arrays(ci, pi, ob, cams, pts)
    ref = oracle_mod.solve(p.num_cameras(), p.num_points(), p.camera_index(), p.point_index(), p.observations(),
                           p.cameras(), p.points(), oracle_mod.default_options(**FIXED))
    out = S.SolveBA(p, linear_solver=C.SOLVER_DENSE_SCHUR, **FIXED)
    # as above: at most 1e7 in condition times unit roundoff, per step
    assert abs(out["final_cost"] - ref["final_cost"]) <= 1e-8 * ref["final_cost"]
    np.testing.assert_allclose(p.cameras(), ref["cams"], rtol=0, atol=1e-7 * np.abs(ref["cams"]).max())


# A camera without observations and without damping: its pivots are exactly zero, in each step of the
# factorization that its place can fall into.  Every step is refused, the parameters stay.
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("nc,unused", [(12, 5), (24, 23), (40, 0), (40, 9), (60, 31), (116, 110)])
def test_dense_zero_pivots_refuse_the_step(oracle_mod, nc, unused, mixed):
    p = S.synthetic(2, seed=nc, num_cameras=nc - 1, num_points=40 * nc, max_track=8)
    ci = p.camera_index() + (p.camera_index() >= unused).astype(np.int32)
    cams = np.insert(p.cameras().reshape(-1, 9), unused, p.cameras()[:9], axis=0)
    q = S.BALProblem.from_arrays(ci, p.point_index(), p.observations().reshape(-1, 2), cams, p.points())
    kw = dict(FIXED, max_num_iterations=20, min_lm_diagonal=1e-300, initial_trust_region_radius=1e60,
              max_trust_region_radius=1e60)  # the damping of a zero column, 1e-360, is zero
    ref = oracle_mod.solve(nc, q.num_points(), ci, p.point_index(), p.observations(), cams.reshape(-1), p.points(),
                           oracle_mod.default_options(**kw))
    assert not any(t["step_is_successful"] for t in ref["trace"][1:])
    out = S.SolveBA(q, linear_solver=C.SOLVER_DENSE_SCHUR, precision=C.PRECISION_MIXED if mixed else C.PRECISION_FP64, **kw)
    assert out["num_successful_steps"] == 0 and out["final_cost"] == out["initial_cost"]
    assert len(out["trace"]) > 1 and not any(t["step_is_successful"] for t in out["trace"][1:])
    np.testing.assert_array_equal(q.cameras(), cams.reshape(-1))
    np.testing.assert_array_equal(q.points(), p.points())
