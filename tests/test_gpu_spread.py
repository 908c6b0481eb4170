"""Small batches of the lane-group layout: path counts at which the groups of a wave that take paths,
or the kernel instance, change; against the oracle.  Per-lane layout: spread over up to one wave per
CU, path counts around the points where the lanes of a wave
that take paths change (1 up to one path per CU, 64 from 64 paths per CU on)."""
import numpy as np
import pytest

import oracle
import systems
from hcgpu.configs import cgauss, sparse_param_system
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


@pytest.mark.parametrize("n,npaths", [(3, 5), (3, 1023), (3, 1025), (3, 4097), (18, 3), (18, 1025), (18, 2050)])
def test_group_batch_sizes(gpu_ctx, n, npaths):
    """One to four 16-lane groups per wave; one or two 32-lane groups per wave, with one and with two
    workgroups per CU."""
    rng = np.random.default_rng(n + npaths)
    F = sparse_param_system(n, 4, n + 2, seed=n)
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
    Q = p0 + 0.05 * cgauss(rng, 9, n + 2)
    H = ParameterHomotopy(F, p0, Q, lift_affine=True)
    g = (np.arange(npaths) % 9).astype(np.int32)
    out = track_batch(gpu_ctx.program(H, layout="group"), np.tile(x0, (npaths, 1)), make_options(), group_of_path=g)
    ref = oracle.track_batch(H, np.tile(x0, (9, 1)), make_options(), group_of_path=np.arange(9, dtype=np.int32))
    np.testing.assert_array_equal(out.code, ref.code[g])
    np.testing.assert_array_equal(out.accepted_steps, ref.accepted_steps[g])
    np.testing.assert_array_equal(out.solution, ref.solution[g])


def test_launch_info_follows_the_instance(gpu_ctx):
    """17 to 24 variables: a launch of at most one workgroup per CU takes the instance with more registers."""
    F = sparse_param_system(18, 4, 20, seed=18)
    H = ParameterHomotopy(F, np.zeros(20), [np.zeros(20)], lift_affine=True)
    p = gpu_ctx.program(H, layout="group")
    cus = p.kernel_info()["cus"]
    small, large = p.launch_info(2 * 4 * cus), p.launch_info(2 * 4 * cus + 1)
    assert (small["workgroups"], large["workgroups"]) == (cus, cus + 1)
    assert small["vgprs"] > large["vgprs"] and large["vgprs"] == p.kernel_info()["vgprs"]
    assert (small["waves_per_simd_built"], large["waves_per_simd_built"]) == (1, 2)
