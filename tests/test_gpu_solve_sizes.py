"""Per-lane tracker at the sizes where its solves change form: n = 1 (no factorization), n = 9 (matrix
held in registers; with two waves per SIMD columns read again), n = 11 and 12 (columns read again),
n = 13 (in memory).  Every path equals the oracle's, bit for bit."""
import numpy as np
import pytest

import oracle
from hcgpu.configs import solve_size_homotopy
from hcgpu.gpu import track_batch
from hcgpu.solve import make_options

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,waves", [(1, 1), (9, 1), (9, 2), (11, 1), (12, 1), (13, 1)])
def test_per_lane_equals_oracle(gpu_ctx, n, waves):
    H, x0 = solve_size_homotopy(n)
    S = np.tile(x0, (9, 1))
    g = np.arange(9, dtype=np.int32)
    out = track_batch(gpu_ctx.program(H, waves_per_eu=waves, layout="lane"), S, make_options(), group_of_path=g)
    ref = oracle.track_batch(H, S, make_options(), group_of_path=g)
    for f in ("code", "accepted_steps", "rejected_steps", "newton_iters", "accuracy", "omega", "mu", "cond"):
        np.testing.assert_array_equal(getattr(out, f), getattr(ref, f), err_msg=f)
    np.testing.assert_array_equal(out.solution, ref.solution)
    assert (out.code == 1).any()
