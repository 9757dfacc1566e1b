"""eval_cost at the sizes where its path changes: cameras in one block's LDS (up to 256) or gathered from
memory, a last block of one observation, more observations than the largest grid takes in one turn."""
import numpy as np
import pytest

import slamplay_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,no", [(1, 1), (1, 257), (256, 4096), (257, 4097), (300, 1), (255, 600001), (900, 524289)])
def test_cost_sizes_match_oracle(oracle_mod, nc, no):
    rng = np.random.default_rng(nc + no)
    npt = max(1, no // 7)
    cams = np.concatenate([rng.normal(0, 0.3, (nc, 3)), rng.normal(0, 0.5, (nc, 2)), rng.normal(-12, 0.5, (nc, 1)),
                           rng.normal(500, 20, (nc, 1)), rng.normal(0, 1e-3, (nc, 2))], axis=1)
    cams[0, :3] = 0.0  # the first-order rotation branch
    if nc > 2:
        cams[1, :3] = [1e-9, -2e-9, 1e-9]
    pts = rng.normal(0, 1.5, (npt, 3))
    ci, pi = rng.integers(0, nc, no).astype(np.int32), rng.integers(0, npt, no).astype(np.int32)
    obs = rng.normal(0, 60, (no, 2))
    p = S.BALProblem.from_arrays(ci, pi, obs, cams, pts)
    for loss, scale in ((1, 1.0), (1, 40.0), (0, 1.0)):
        ref = oracle_mod.cost(ci, pi, obs, cams, pts, loss, scale)
        # sums of nonnegative FP64 terms in another order, each term within a few dozen roundings
        assert abs(S.eval_cost(p, loss=loss, loss_scale=scale) - ref) <= 1e-12 * ref
