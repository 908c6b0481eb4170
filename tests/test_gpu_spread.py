"""Small batches spread over one wave per CU: path counts around the points where the lanes of a wave
that take paths change (1 up to one path per CU, 64 from 64 paths per CU on)."""
import numpy as np
import pytest

import oracle
import systems
from hcgpu.gpu import track_batch
from hcgpu.homotopies import ParameterHomotopy
from hcgpu.solve import make_options

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npaths", [1, 2, 63, 64, 255, 256, 257, 511, 513, 256 * 63, 256 * 63 + 1, 256 * 64 + 1])
def test_batch_sizes(gpu_ctx, npaths):
    rng = np.random.default_rng(npaths)
    Q = np.array([2, 4]) + 0.3 * (rng.standard_normal((7, 2)) + 1j * rng.standard_normal((7, 2)))
    H = ParameterHomotopy(systems.tracker_param_system(), [1, 0], Q)
    S = np.array([[1, 1], [-1, -1]], dtype=complex)[np.arange(npaths) % 2]
    g = (np.arange(npaths) % 7).astype(np.int32)
    out = track_batch(gpu_ctx.program(H), S, make_options(), group_of_path=g)
    ref = oracle.track_batch(H, S, make_options(), group_of_path=g)
    np.testing.assert_array_equal(out.code, ref.code)
    np.testing.assert_array_equal(out.accepted_steps, ref.accepted_steps)
    np.testing.assert_array_equal(out.solution, ref.solution)  # the arithmetic is fixed, bit for bit
    assert gpu_ctx.last_counters()["steps"] == int((ref.accepted_steps + ref.rejected_steps).sum())
