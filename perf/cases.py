"""Performance cases: the calls that programs built on this framework make, over their real range of
sizes, each through a public entry point.

Tracking cases return every output of the call: the records' whole numbers and floating fields, the
endpoints, last points and valuations.  The tracker is a deterministic function of its inputs whose
arithmetic is fixed operation by operation (the layouts and the CPU oracle agree bit for bit), so two
correct builds return the same bits and the tolerance is "exact".  Training sums gradients over blocks in
an order that the arithmetic does not fix, and has a tolerance of its own.
"""
import ctypes
import functools
import math
import sys
from pathlib import Path

import numpy as np
import torch  # before the library: one HIP runtime per process

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "homotopycontinuation.jl_amd"))

from hcgpu import learned  # noqa: E402
from hcgpu.abi import hcg_path_result  # noqa: E402
from hcgpu.configs import cfg2_problem, cfg4_problem, cgauss, dense_system, parameter_draws, sparse_param_system  # noqa: E402
from hcgpu.device import DeviceBatch  # noqa: E402
from hcgpu.gpu import GpuContext, track_batch, track_multi  # noqa: E402
from hcgpu.homotopies import ParameterHomotopy, total_degree  # noqa: E402
from hcgpu.polys import System, variables  # noqa: E402
from hcgpu.solve import make_options  # noqa: E402

NMIXED = (4, 6, 8, 12)


def listed():
    return [
        # one path of a two-variable parameter homotopy: the interactive `track(tracker, x)`, all latency
        dict(name="track_one_path", kind="pair", paths=1, via="host"),
        # a total-degree solve of dense quartic size: two waves, as slow as its longest path
        dict(name="dense4_solve", kind="dense", n=4, paths=81, via="host"),
        # all 1,024 solutions moved to one new parameter value, the serving call, from host arrays
        dict(name="param10_one_target", kind="param10", targets=1, paths=1024, learned=False, via="host"),
        # the same solutions moved to a ragged number of targets, replayed from a captured graph
        dict(name="param10_graph", kind="param10", targets=17, paths=16391, learned=True, via="graph"),
        # many_solve over 61 targets with the plain step rule
        dict(name="param10_plain", kind="param10", targets=61, paths=61777, learned=False, via="device"),
        # many_solve over 256 targets with the learned step: the largest batch
        dict(name="param10_learned", kind="param10", targets=256, paths=262144, learned=True, via="device"),
        # total-degree solve of dense cubics, wide rows and few waves
        dict(name="dense8_solve", kind="dense", n=8, paths=6561, via="device"),
        # systems of several sizes in one launch, most paths diverging (endgame decides at infinity)
        dict(name="mixed_learned", kind="mixed", paths12=30011, learned=True, via="host"),
        # fifteen variables, past the size where a path fits a lane: one solution carried to many targets
        dict(name="sparse15_targets", kind="sparse", n=15, paths=2048, via="device"),
        # twenty-two variables: groups of half a wave
        dict(name="sparse22_targets", kind="sparse", n=22, paths=601, via="host"),
        # certificates for the endpoints of a many-parameter solve
        dict(name="certify_endpoints", kind="certify", targets=16, candidates=16000),
        # training of the step proposer on logged steps: forward, backward and optimizer
        dict(name="train_proposer", kind="train", records=200003, epochs=1, batch=4096),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["pair", "dense", "param10", "param10", "param10", "mixed", "sparse", "sparse", "certify", "train"])
    if kind == "pair":
        return dict(kind=kind, paths=_log_int(rng, 1, 3000), via=rng.choice(["host", "device"]))
    if kind == "dense":
        n = rng.choice([4, 8])
        return dict(kind=kind, n=n, paths=_log_int(rng, 5, 3**n), via=rng.choice(["host", "device", "graph"]))
    if kind == "param10":
        plain = rng.random() < 0.5  # the plain rule takes about twice the learned rule's time
        paths = _log_int(rng, 30, 110000 if plain else 230000)
        return dict(kind=kind, targets=-(-paths // 1024), paths=paths, learned=not plain,
                    via=rng.choice(["host", "device", "graph"]))
    if kind == "mixed":
        plain = rng.random() < 0.5
        return dict(kind=kind, paths12=_log_int(rng, 500, 12000 if plain else 28000), learned=not plain, via="host")
    if kind == "sparse":
        n = rng.randint(13, 24)
        return dict(kind=kind, n=n, paths=_log_int(rng, 8, 2000 if n <= 16 else 600), via=rng.choice(["host", "device"]))
    if kind == "certify":
        c = _log_int(rng, 100, 40000)
        return dict(kind=kind, targets=-(-c // 1000), candidates=c)
    return dict(kind=kind, records=_log_int(rng, 3000, 300000), epochs=rng.choice([1, 2]), batch=rng.choice([1024, 4096]))


# ------------------------------ the problems ------------------------------
# Systems and their lowering are fixed parts of a user's program, the same for every seed; the
# programs made from them are kept per process, as such a program keeps them.


@functools.lru_cache(maxsize=None)
def _pair_system():
    (x, y), (a, b) = variables(2, 2)
    return System([x**2 - a, x * y - a + b], 2, 2)


@functools.lru_cache(maxsize=None)
def _dense(n):
    return dense_system(n, 3, seed=100 if n == 4 else 1)


@functools.lru_cache(maxsize=None)
def _sparse(n):
    """(F, x0, p0): sparse quadrics with n + 6 parameters and one solution x0 at p0.  The system is
    linear in its parameters, so p0 is the least-norm solution of a linear system."""
    F = sparse_param_system(n, 20, n + 6, seed=60 + n)
    rng = np.random.default_rng(60 + n)
    x0 = cgauss(rng, n)
    A, b = np.zeros((n, n + 6), dtype=complex), np.zeros(n, dtype=complex)
    for i, f in enumerate(F.polys):
        for e, c in f.terms.items():
            m = complex(c) * np.prod(x0 ** np.array(e[:n]))
            if any(e[n:]):
                A[i, e[n:].index(1)] += m
            else:
                b[i] -= m
    return F, x0, np.linalg.lstsq(A, b, rcond=None)[0]


@functools.lru_cache(maxsize=None)
def _context(key):
    """One context with one program, made once: (context, program, homotopy, extra)."""
    ctx = GpuContext(0)
    if key[0] == "pair":
        H, extra = ParameterHomotopy(_pair_system(), [1, 0], [2, 4]), None
    elif key[0] == "dense":
        H, extra = total_degree(_dense(key[1]), seed=101 if key[1] == 4 else 2)
    elif key[0] == "param10":
        F, p0, Q = cfg2_problem(256)
        H, extra = ParameterHomotopy(F, p0, Q, lift_affine=True), np.load(ROOT / "tests" / "golden" / "cfg2_starts.npy")
        learned.load(ctx, learned.saved_weights("param10_step_mlp"))
    elif key[0] == "mixed":
        probs = cfg4_problem(NMIXED)
        learned.load(ctx, learned.saved_weights("mixed_step_mlp"))
        return ctx, ctx.program_multi([h for h, _ in probs]), [h for h, _ in probs], [s for _, s in probs]
    elif key[0] == "sparse":
        F, x0, p0 = _sparse(key[1])
        H, extra = ParameterHomotopy(F, p0, [p0], lift_affine=True), x0
    elif key[0] == "certify":
        F, _, _ = cfg2_problem(1)
        return ctx, ctx.certifier(F), F, None
    else:
        return ctx, None, None, None
    return ctx, ctx.program(H), H, extra


# --------------------------------- inputs ---------------------------------


def _track_inputs(case, seed):
    """(starts, target parameters or None, group of each path or None) on the host."""
    rng = np.random.default_rng([seed, 77])
    kind, P = case["kind"], case["paths"]
    if kind == "pair":
        S = np.array([[1, 1], [-1, -1]], dtype=complex)[np.arange(P) % 2]
        return S, np.array([2, 4]) + 0.5 * cgauss(rng, P, 2), np.arange(P, dtype=np.int32)
    if kind == "dense":  # a solve tracks all starts; another seed takes them in another order
        S = _context(("dense", case["n"]))[3]
        return S[rng.permutation(len(S))[:P]], None, None
    if kind == "param10":
        S = _context(("param10",))[3]
        Q = parameter_draws(16, case["targets"], seed=seed + 1000)
        g = np.repeat(np.arange(case["targets"], dtype=np.int32), len(S))[:P]
        return np.tile(S, (case["targets"], 1))[:P], Q, g
    F, x0, p0 = _sparse(case["n"])
    return np.tile(x0, (P, 1)), p0 + cgauss(rng, P, len(p0)) * np.abs(p0).max(), np.arange(P, dtype=np.int32)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("pair", "dense", "param10", "sparse"):
        key = (kind, case["n"]) if "n" in case else (kind,)
        ctx, prog, H, _ = _context(key)
        S, Q, g = _track_inputs(case, seed)
        T = None if Q is None else H.target_matrix(Q)
        opts = make_options(learned_step=1) if case.get("learned") else make_options()
        if case["via"] == "host":
            return dict(do="host", prog=prog, starts=S, targets=T, groups=g, opts=opts)
        batch = DeviceBatch(ctx, prog, S, None if T is None else H.p, T, g)
        return dict(do=case["via"], batch=batch, opts=opts, graph=batch.graph(opts) if case["via"] == "graph" else None)
    if kind == "mixed":
        ctx, prog, Hs, Ss = _context(("mixed",))
        rng = np.random.default_rng([seed, 78])
        starts = [S[rng.permutation(len(S))[:case["paths12"] if n == 12 else len(S)]] for n, S in zip(NMIXED, Ss)]
        return dict(do="multi", prog=prog, starts=starts, opts=make_options(learned_step=1 if case["learned"] else 0))
    if kind == "certify":
        # endpoints as a solver or a file hands them over, correct to about ten digits
        ctx, cert, F, _ = _context(("certify",))
        _, prog, H, S = _context(("param10",))
        C, T = case["candidates"], case["targets"]
        Q = parameter_draws(16, T, seed=seed + 1000)
        g = np.arange(C, dtype=np.int32) % T
        X = track_batch(prog, S[(np.arange(C) // T) % len(S)], make_options(learned_step=1), target_groups=H.target_matrix(Q),
                        group_of_path=g).solution
        X = np.round(X * 2.0**33) / 2.0**33
        return dict(do="certify", cert=cert, X=X, Q=Q, groups=g)
    rng = np.random.default_rng([seed, 79])
    N = case["records"]
    X = rng.standard_normal((N, 8)).astype(np.float32)  # features are scaled to zero mean and unit variance
    Y = np.stack([0.6 * X[:, 0] - 0.3 * np.tanh(X[:, 2] * X[:, 5]) + 0.1 * rng.standard_normal(N),
                  (X[:, 3] + X[:, 6] > 1).astype(np.float64)], axis=1).astype(np.float32)
    W = np.stack([rng.random(N) < 0.9, np.ones(N)], axis=1).astype(np.float32)
    return dict(do="train", ctx=_context(("train",))[0], p=learned.init_params(seed), X=X, Y=Y, W=W, epochs=case["epochs"],
                batch=case["batch"])


# ---------------------------------- a pass ----------------------------------

_INTS = [f for f, t in hcg_path_result._fields_ if t is ctypes.c_int32]
_FLOATS = [f for f, t in hcg_path_result._fields_ if t is not ctypes.c_int32]


def _host(o):
    out = {f: o.records[f] for f in _INTS + _FLOATS}
    out.update(solution=o.solution, last_point=o.last_point, valuation=o.valuation)
    return out


def run(state):
    do = state["do"]
    if do == "host":
        return _host(track_batch(state["prog"], state["starts"], state["opts"], state["targets"], state["groups"]))
    if do in ("device", "graph"):
        b = state["batch"]
        if do == "graph":
            state["graph"].launch()
        else:
            b.launch(state["opts"])
        ni, nf = len(_INTS), len(_FLOATS)
        return dict(counts=b.res.view(torch.int32).view(b.npaths, ni + 2 * nf)[:, :ni],
                    values=b.res.view(torch.float64).view(b.npaths, ni // 2 + nf)[:, ni // 2:],
                    solution=b.sol, last_point=b.last, valuation=b.val)
    if do == "multi":
        outs = track_multi(state["prog"], state["starts"], state["opts"])
        return [dict(code=o.code, singular=o.singular, steps=o.accepted_steps + o.rejected_steps, cond=o.cond, solution=o.solution,
                     last_point=o.last_point, valuation=o.valuation) for o in outs]
    if do == "certify":
        o = state["cert"].certify(state["X"], state["Q"], real_system=False, group_of=state["groups"])
        out = {f: o.records[f] for f in o.records.dtype.names}
        out.update(box1=o.box1, box0=o.box0, refined=o.refined)
        return out
    p, loss = learned.train(state["ctx"], state["p"], state["X"], state["Y"], state["W"], epochs=state["epochs"],
                            batch=state["batch"])
    return dict(params=p, loss=loss)


# ------------------------- what a pass cannot do without -------------------------

# counted FP64 flops of one tracker step and steps of one path, as the tracker's own counters report
# them (plain step rule; the learned rule takes about half the steps, each a little dearer)
_STEP = {"pair": (900, 12), "dense4": (9200, 50), "dense8": (240959, 72.4), "param10": (69900, 83.7), "param10_learned": (72000, 38.6),
         "mixed12": (331790, 90.5), "mixed12_learned": (350000, 48.0)}


def work(case):
    kind = case["kind"]
    if kind == "train":
        N = case["records"] * case["epochs"]
        return dict(bytes=N * 4.0 * (8 + 2 + 2), flops=3.0 * 9472 * N)
    if kind == "certify":
        C, n = case["candidates"], 10
        return dict(bytes=C * (16.0 * n * 2 + 40 + 64 * n + 4) + case["targets"] * 256, flops=C * 6.0e4)
    if kind == "mixed":
        k = "mixed12_learned" if case["learned"] else "mixed12"
        P = case["paths12"]
        return dict(bytes=P * (104.0 + 56 * 12) + 7371 * (104.0 + 56 * 8), flops=P * _STEP[k][0] * _STEP[k][1] + 7371 * 4.0e6)
    P = case["paths"]
    n = case.get("n", 2 if kind == "pair" else 10)
    if kind == "sparse":  # evaluation, factorization and solves of a step
        f, s = 4 * (11 * n * (n - 1) / 2 + 8 * (n - 1) * n * (2 * n - 1) / 6 + 600 * n) + 7 * (8 * n * (n - 1) + 11 * n), 60
    else:
        f, s = _STEP["param10_learned" if case.get("learned") else kind + str(n) if kind == "dense" else kind]
    return dict(bytes=P * (104.0 + 56 * n) + (P * 16.0 * n if kind == "sparse" else 0), flops=P * f * float(s))


def tolerance(case):
    if case["kind"] != "train":
        return "exact"
    # Weights are rounded to bf16 in the forward pass and Adam divides by the root of the squared gradient,
    # so a last-bit difference of one sum grows from step to step.  Four times what FP32 sums in two orders
    # (and FP32 against FP64 sums) differed by: 3.4e-6 after 49 steps, 4.7e-5 after 98, 1.7e-3 after 586;
    # the largest single weight about twelve times that.
    steps = case["epochs"] * -(-case["records"] // case["batch"])
    rel = 1.5e-5 * max(1.0, steps / 49) ** 2.7
    return {"rel": rel, "max": 15 * rel}


# ------------------------------ plain 64-bit results ------------------------------
# The endpoints of the smaller batches by a plain predictor-corrector in numpy: c(t) = t c1 + (1 - t) c0 on
# a common list of monomials, tangent by a linear solve, Heun's predictor, Newton's corrector, a step for
# each path.  Larger batches would take minutes here.


def _table(polys, n):
    """(equation, exponents) of every monomial of a list of {exponents: coefficient}."""
    keys = sorted({(i, e) for i, f in enumerate(polys) for e in f})
    return keys


class _Coefficients:
    """F(x, c) and its derivatives for monomials of degree at most 3, as products of three entries of (1, x)."""

    def __init__(self, keys, n):
        self.n = n

        def factors(e, m):
            v = [k + 1 for k in range(n) for _ in range(e[k])]
            return v + [0] * (m - len(v))

        self.mon = np.array([factors(e, 3) for _, e in keys])
        self.to_eq = np.zeros((len(keys), n))
        self.to_eq[np.arange(len(keys)), [i for i, _ in keys]] = 1
        rows = [(k, e[j], factors(tuple(v - (m == j) for m, v in enumerate(e)), 2), i * n + j)
                for k, (i, e) in enumerate(keys) for j in range(n) if e[j]]
        self.dk = np.array([r[0] for r in rows])
        self.df = np.array([float(r[1]) for r in rows])
        self.dmon = np.array([r[2] for r in rows])
        self.to_jac = np.zeros((len(rows), n * n))
        self.to_jac[np.arange(len(rows)), [r[3] for r in rows]] = 1

    def value(self, x, c):
        z = np.concatenate([np.ones((len(x), 1)), x], axis=1)
        a, b, d = self.mon.T
        return (c * z[:, a] * z[:, b] * z[:, d]) @ self.to_eq

    def jacobian(self, x, c):
        z = np.concatenate([np.ones((len(x), 1)), x], axis=1)
        a, b = self.dmon.T
        return ((c[:, self.dk] * self.df * z[:, a] * z[:, b]) @ self.to_jac).reshape(len(x), self.n, self.n)


def _endpoints(tab, c1, c0, x):
    """Endpoints at t = 0 of the paths that start in x at t = 1 (c1 and c0: a row for each path)."""
    def at(t, rows):
        return t[:, None] * c1[rows] + (1 - t[:, None]) * c0[rows]

    def solve(x, t, rows, rhs):
        return np.linalg.solve(tab.jacobian(x, at(t, rows)), rhs[..., None])[..., 0]

    x, t, h = x.copy(), np.ones(len(x)), np.full(len(x), 0.01)
    rows = np.arange(len(x))
    while len(rows):
        X, T = x[rows], t[rows]
        H = np.minimum(h[rows], T)
        rate = c1[rows] - c0[rows]
        v1 = solve(X, T, rows, tab.value(X, rate))
        v2 = solve(X + H[:, None] * v1, T - H, rows, tab.value(X + H[:, None] * v1, rate))
        Z = X + H[:, None] * (v1 + v2) / 2
        first = None
        for _ in range(3):
            d = solve(Z, T - H, rows, tab.value(Z, at(T - H, rows)))
            Z = Z - d
            last = np.abs(d).max(axis=1) / np.abs(Z).max(axis=1)
            first = last if first is None else first
        good = (first < 2e-4) & (last < 1e-11)
        x[rows[good]], t[rows[good]] = Z[good], (T - H)[good]
        h[rows] = np.where(good, np.where(first < 2e-5, 1.6, 1.0) * H, H / 2)
        rows = rows[t[rows] > 0]
        if len(rows) and h[rows].min() < 1e-9:
            return None
    for _ in range(3):
        x = x - solve(x, t, np.arange(len(x)), tab.value(x, c0))
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("pair", "dense", "param10", "sparse") or case["paths"] * case.get("n", 10 if kind == "param10" else 2) > 400:
        return None
    S, Q, g = _track_inputs(case, seed)
    n, P = S.shape[1], len(S)
    if kind == "dense":
        H = _context(("dense", n))[2]
        F = [f.terms for f in _dense(n).polys]
        keys = _table(F, n)
        c0 = np.array([F[i][e] for i, e in keys])
        c1 = np.zeros(len(keys), dtype=complex)
        for i, f in enumerate(F):  # gamma s (x_i^3 - 1)
            s = H.gamma * max(abs(c) for c in f.values())
            c1[keys.index((i, tuple(3 * (k == i) for k in range(n))))] = s
            c1[keys.index((i, (0,) * n))] = -s
        C1, C0 = np.tile(c1, (P, 1)), np.tile(c0, (P, 1))
    else:
        if kind == "pair":
            F, p0 = _pair_system(), np.array([1, 0])
        elif kind == "param10":
            F, p0, _ = cfg2_problem(1)
        else:
            F, _, p0 = _sparse(n)
        terms = [f.terms for f in F.polys]
        keys = sorted({(i, e[:n]) for i, f in enumerate(terms) for e in f})
        A, b = np.zeros((len(keys), len(p0)), dtype=complex), np.zeros(len(keys), dtype=complex)
        for i, f in enumerate(terms):  # every coefficient is affine in the parameters
            for e, c in f.items():
                k = keys.index((i, e[:n]))
                if any(e[n:]):
                    A[k, e[n:].index(1)] += c
                else:
                    b[k] += c
        C1, C0 = np.tile(A @ p0 + b, (P, 1)), (np.asarray(Q) @ A.T + b)[g]
    x = _endpoints(_Coefficients(keys, n), C1, C0, S.astype(complex))
    if x is None:
        return None
    return dict(solution=x) if case["via"] == "host" else dict(solution=torch.from_numpy(x.view(np.float64).reshape(-1)))
