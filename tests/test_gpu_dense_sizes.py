"""The dense reduced system at the sizes where its kernels change path: one tile of 32 unknowns, exact
tile multiples, one tile past a 512-row block of the triangular solves and of its second block."""
import numpy as np
import pytest

import slamplay_amd as S
from slamplay_amd import _capi as C

pytestmark = pytest.mark.gpu

FIXED = dict(max_num_iterations=3, function_tolerance=0.0, gradient_tolerance=0.0, parameter_tolerance=0.0)


# 9 nc unknowns: 27, 36, 63, 180, 189, 198 (one workgroup, tiles of 32 columns), 288 and 297 (64 x 64 blocks: 4 and a
# half, and a little more), 513 and 1026 (one and two 512-row blocks of the sweeps and the first of another)
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


def _against_oracle(oracle_mod, nc, mixed, **kw):
    p = S.synthetic(2, seed=nc, num_cameras=nc, num_points=40 * nc, max_track=min(8, nc))
    ref = oracle_mod.solve(p.num_cameras(), p.num_points(), p.camera_index(), p.point_index(), p.observations(),
                           p.cameras(), p.points(), oracle_mod.default_options(**kw))
    out = S.SolveBA(p, linear_solver=C.SOLVER_DENSE_SCHUR, precision=C.PRECISION_MIXED if mixed else C.PRECISION_FP64, **kw)
    assert out["num_successful_steps"] == sum(t["step_is_successful"] for t in ref["trace"][1:])
    return out, ref, p


# Past one workgroup's 198 unknowns the system is padded to 64 x 64 blocks: 207 unknowns (the first), 576 and 1152 (9
# and 18 blocks exactly), 639 (one short of 10); the sweeps' blocks of 512 rows end inside the first of them
# and after 8 and 16 blocks.
@pytest.mark.parametrize("nc", [23, 64, 71, 128])
def test_dense_block_edges_match_oracle(oracle_mod, nc):
    out, ref, p = _against_oracle(oracle_mod, nc, False, **FIXED)
    # as above: at most 1e7 in condition times unit roundoff, per step
    assert abs(out["final_cost"] - ref["final_cost"]) <= 1e-8 * ref["final_cost"]
    np.testing.assert_allclose(p.cameras(), ref["cams"], rtol=0, atol=1e-7 * np.abs(ref["cams"]).max())


# The FP32 factor (from 289 unknowns on) at the same edges and at 297, 513 and 1026 (4, 8 and 16 blocks and
# something).  Well damped, so that the steps are the factor's and not the rounding of the FP32 Jacobians along
# weak directions: D^2 is the diagonal, a third and a ninth of it.
@pytest.mark.parametrize("nc", [33, 57, 64, 71, 114, 128])
def test_dense_mixed_block_edges_match_oracle(oracle_mod, nc):
    start = S.synthetic(2, seed=nc, num_cameras=nc, num_points=40 * nc, max_track=min(8, nc)).cameras().copy().reshape(-1, 9)
    out, ref, p = _against_oracle(oracle_mod, nc, True, **dict(FIXED, initial_trust_region_radius=1.0))
    # FP32 Jacobian entries are right to 1e-5 (roundings of 6e-8 and the cancellation in a projection), the condition
    # of the damped, scaled system is at most 100: 1e-3 of the step in each kind of parameter, and so of the
    # decrease
    step = np.abs(ref["cams"].reshape(-1, 9) - start).max(axis=0)
    assert (np.abs(p.cameras().reshape(-1, 9) - ref["cams"].reshape(-1, 9)).max(axis=0) <= 1e-3 * step).all()
    assert abs(out["final_cost"] - ref["final_cost"]) <= 1e-3 * (ref["initial_cost"] - ref["final_cost"])
