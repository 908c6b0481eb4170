"""Per-lane tracker at the sizes where its solves change form: n = 1 (no factorization), n = 9 (matrix
held in registers; with two waves per SIMD columns read again), n = 11 and 12 (columns read again),
n = 13 (in memory).  Every path equals the oracle's, bit for bit."""
import numpy as np
import pytest

import oracle
from hcgpu.configs import cgauss, sparse_param_system
from hcgpu.gpu import track_batch
from hcgpu.homotopies import ParameterHomotopy
from hcgpu.solve import make_options

pytestmark = pytest.mark.gpu


def homotopy(n):
    """(H, x0): sparse quadrics with one solution x0 at the start parameters, and nine targets."""
    rng = np.random.default_rng(n)
    F = sparse_param_system(n, 3 if n == 1 else 4, n + 2, seed=n)
    x0 = cgauss(rng, n)
    A, b = np.zeros((n, n + 2), dtype=complex), np.zeros(n, dtype=complex)
    for i, f in enumerate(F.polys):  # p0 with F(x0; p0) = 0: the coefficients are affine in the parameters
        for e, c in f.terms.items():
            m = complex(c) * np.prod(x0 ** np.array(e[:n]))
            if any(e[n:]):
                A[i, e[n:].index(1)] += m
            else:
                b[i] -= m
    p0 = np.linalg.lstsq(A, b, rcond=None)[0]
    return ParameterHomotopy(F, p0, p0 + 0.3 * cgauss(rng, 9, n + 2), lift_affine=True), x0


@pytest.mark.parametrize("n,waves", [(1, 1), (9, 1), (9, 2), (11, 1), (12, 1), (13, 1)])
def test_per_lane_equals_oracle(gpu_ctx, n, waves):
    H, x0 = homotopy(n)
    S = np.tile(x0, (9, 1))
    g = np.arange(9, dtype=np.int32)
    out = track_batch(gpu_ctx.program(H, waves_per_eu=waves, layout="lane"), S, make_options(), group_of_path=g)
    ref = oracle.track_batch(H, S, make_options(), group_of_path=g)
    for f in ("code", "accepted_steps", "rejected_steps", "newton_iters", "accuracy", "omega", "mu", "cond"):
        np.testing.assert_array_equal(getattr(out, f), getattr(ref, f), err_msg=f)
    np.testing.assert_array_equal(out.solution, ref.solution)
    assert (out.code == 1).any()
