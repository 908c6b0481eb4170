"""Certifiers whose tapes split at their parameter-only coefficients (evaluated once per parameter
vector): records and boxes equal the oracle's, which evaluates the whole tapes, bit for bit."""
import numpy as np
import pytest

import oracle
from hcgpu.certify import parameter_boxes
from hcgpu.configs import cgauss, parameter_product_system, sparse_param_system
from hcgpu.homotopies import _SysTapes

pytestmark = pytest.mark.gpu


def system(name):
    if name == "affine3":  # 72 coefficient operations, affine in four parameters
        return sparse_param_system(3, 6, 4, seed=7)
    return parameter_product_system()


def _zeros(F, q, rng):
    """A few zeros of F(.; q) by Newton's method from random points, in plain complex128."""
    f = [[(c, e) for e, c in g.terms.items()] for g in F.polys]

    def val(x):
        z = np.concatenate([x, q])
        return np.array([sum(c * np.prod(z ** np.array(e)) for c, e in g) for g in f])

    out = []
    while len(out) < 6:
        x = cgauss(rng, 3)
        for _ in range(60):
            J = np.stack([(val(x + 1e-7 * d) - val(x - 1e-7 * d)) / 2e-7 for d in np.eye(3)], axis=1)
            x = x - np.linalg.solve(J, val(x))
        if np.abs(val(x)).max() < 1e-9 and np.abs(x).max() < 1e3:
            out.append(x)
    return np.array(out)


@pytest.mark.parametrize("name", ["affine3", "products3"])
@pytest.mark.parametrize("ngroups", [1, 5])
def test_split_equals_whole(gpu_ctx, name, ngroups):
    F = system(name)
    rng = np.random.default_rng(3 + ngroups)
    Q = cgauss(rng, ngroups, 4)
    X = np.concatenate([_zeros(F, q, rng) for q in Q])
    X[::4] += 1e-3  # some candidates that are no zeros, so that the extended retry runs too
    X[::4] *= 1.5
    G = np.repeat(np.arange(ngroups, dtype=np.int32), 6)
    enc = [parameter_boxes(list(q)) for q in Q]
    P, I, B = (np.stack([e[k] for e in enc]) for k in range(3))
    I[:, :, [0, 2]] -= 1e-13  # parameter boxes and balls of some width
    I[:, :, [1, 3]] += 1e-13
    B[:, :, [2, 5]] += 1e-30
    cert = gpu_ctx.certifier(F)
    assert "#define HCG_CERT_NCE 0\n" not in cert.source()
    tapes = _SysTapes(F)
    for refine in (True, False):
        g = cert.certify(X, P, I, B, refine=refine, real_system=False, group_of=G)
        o = oracle.certify(tapes.struct(), 3, X, P, I, B, refine, True, False, 4, group_of=G)
        for f in ("certified", "real", "complex_", "newton_iters", "prec", "contraction", "inflation"):
            np.testing.assert_array_equal(getattr(g, f), getattr(o, f), err_msg=f)
        np.testing.assert_array_equal(g.box1, o.box1)
        np.testing.assert_array_equal(g.box0, o.box0)
        np.testing.assert_array_equal(g.refined, o.refined)
    assert g.certified.any()


@pytest.mark.parametrize("name,nsol,ngroups", [("affine3", 12014, 12014), ("affine3", 12015, 12015), ("products3", 4372, 4372),
                                               ("products3", 4373, 4373), ("products3", 9000, 4661), ("products3", 9000, 4662)])
def test_tables_or_whole_tapes(gpu_ctx, name, nsol, ngroups):
    """The largest number of parameter vectors that takes tables, and the smallest that takes whole
    tapes, with groups out of order; random points, about half of which converge to zeros."""
    F = system(name)
    rng = np.random.default_rng(nsol + ngroups)
    Q, X = cgauss(rng, ngroups, 4), cgauss(rng, nsol, 3)
    G = rng.permutation(np.arange(nsol, dtype=np.int32) % ngroups)
    g = gpu_ctx.certifier(F).certify(X, Q, real_system=False, group_of=G)
    enc = [parameter_boxes(list(q)) for q in Q]
    P, I, B = (np.stack([e[k] for e in enc]) for k in range(3))
    tapes = _SysTapes(F)
    o = oracle.certify(tapes.struct(), 3, X, P, I, B, True, True, False, 16, group_of=G)
    for f in ("certified", "newton_iters", "prec", "contraction", "inflation"):
        np.testing.assert_array_equal(getattr(g, f), getattr(o, f), err_msg=f)
    np.testing.assert_array_equal(g.box1, o.box1)
    np.testing.assert_array_equal(g.refined, o.refined)
    assert 0 < g.certified.sum() < nsol
