"""The work whose speed this repository is measured by: calls of the public
Python entry points over the sizes, precisions and options of the benchmark
configurations and tests.

A program of this framework factors KKT systems whose pattern it analysed once
and whose values change from call to call (SolverSettings, one system or a
batch), solves further right-hand sides with a factor that it keeps, runs
NASOQ's whole active-set loop on quadratic programs (Nasoq), and trains the
network that predicts active sets (ActiveSetPredictor).  The families below
are those calls:

  kkt     new values, factorization, refined solve of one system [H A'; A 0],
          H a 3-D Laplacian, in FP64, FP32 or BF16 factor precision
  indef   the same for block-indefinite matrices, which force 2 x 2 pivots
  batch   the same for many 2-D KKT systems of uneven size in one handle
  solve   further right-hand sides with a factor that is kept
  qp      one whole QP solve (box or general inequality rows)
  mlp     one epoch of training, or the predictions, of the active-set network

prepare() keeps one analysed handle per pattern (the plan such a program keeps);
the seed gives the values and the right-hand sides."""
import functools
import math

import numpy as np
import torch

from nasoq_amd import lbl, learned, qp
from nasoq_amd import problems as P

PRECISION = {"f64": lbl.F64, "f32": lbl.F32, "bf16": lbl.BF16}
DENSE = 6000  # largest order whose dense 64-bit reference takes seconds


def listed():
    return [
        # a test-sized system: one call's latency
        {"name": "kkt5_f64", "family": "kkt", "grid": 5, "rows": 16, "nnz": 6, "nrhs": 1, "precision": "f64",
         "refine": "default"},
        # a small benchmark configuration, the reference's default refinement
        {"name": "kkt16_f64", "family": "kkt", "grid": 16, "rows": 256, "nnz": 8, "nrhs": 1, "precision": "f64",
         "refine": "default"},
        # an ordinary system of odd order with several right-hand sides
        {"name": "kkt33_f64", "family": "kkt", "grid": 33, "rows": 2049, "nnz": 8, "nrhs": 4, "precision": "f64",
         "refine": "target"},
        # the headline configuration
        {"name": "kkt64_f64", "family": "kkt", "grid": 64, "rows": 16384, "nnz": 8, "nrhs": 4, "precision": "f64",
         "refine": "target"},
        # mixed precision: FP32 and BF16 factors with FP64 refinement
        {"name": "kkt48_f32", "family": "kkt", "grid": 48, "rows": 6912, "nnz": 8, "nrhs": 4, "precision": "f32",
         "refine": "target"},
        {"name": "kkt56_bf16", "family": "kkt", "grid": 56, "rows": 10976, "nnz": 8, "nrhs": 4, "precision": "bf16",
         "refine": "target"},
        # dense indefinite blocks with a zero diagonal: 2 x 2 pivots and interchanges
        {"name": "indef24x150_f64", "family": "indef", "blocks": 24, "size": 150, "nrhs": 2, "precision": "f64",
         "refine": "default"},
        # the KKT systems of a batch of QPs of uneven size
        {"name": "batch192_f64", "family": "batch", "count": 192, "lo": 16, "hi": 160, "rows": 64,
         "precision": "f64"},
        # a factor kept for more right-hand sides
        {"name": "solve48_f64", "family": "solve", "grid": 48, "rows": 6912, "nnz": 8, "nrhs": 3, "precision": "f64",
         "refine": "target"},
        # the plain QP configuration (box constraints, equality rows)
        {"name": "qp_box40", "family": "qp", "kind": "box", "grid": 40, "rows": 100},
        # a member of the parametric family whose inequality rows couple six variables each
        {"name": "qp_rows16", "family": "qp", "kind": "rows", "grid": 16, "rows": 102},
        # training the active-set network of the 40 x 40 family
        {"name": "mlp_train", "family": "mlp", "kind": "train", "hidden": 1024, "out": 640, "samples": 384,
         "batch": 64},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    family = rng.choice(["kkt", "kkt", "kkt", "indef", "batch", "solve", "qp", "mlp"])
    if family == "kkt":
        prec = rng.choice(["f64", "f64", "f32", "bf16"])
        g = _log(rng, 5, 62) if prec == "f64" else _log(rng, 12, 62)
        return {"family": family, "grid": g, "rows": max(1, int(g ** 3 / rng.uniform(16, 28))),
                "nnz": rng.randint(6, 8), "nrhs": rng.randint(1, 8), "precision": prec,
                "refine": "target" if prec != "f64" else rng.choice(["default", "target"])}
    if family == "indef":
        return {"family": family, "blocks": _log(rng, 3, 32), "size": _log(rng, 8, 200), "nrhs": rng.randint(1, 8),
                "precision": "f64", "refine": "default"}
    if family == "batch":
        lo = _log(rng, 8, 32)
        hi = _log(rng, lo + 4, 160)
        return {"family": family, "count": _log(rng, 4, max(4, min(256, 5_000_000 // (hi * hi)))), "lo": lo, "hi": hi,
                "rows": rng.randint(8, 64), "precision": rng.choice(["f64", "f64", "f32"])}
    if family == "solve":
        g = _log(rng, 12, 56)
        return {"family": family, "grid": g, "rows": max(1, int(g ** 3 / rng.uniform(16, 28))),
                "nnz": rng.randint(6, 8), "nrhs": rng.randint(1, 8), "precision": "f64",
                "refine": rng.choice(["default", "target"])}
    if family == "qp":
        kind = rng.choice(["box", "rows"])
        g = _log(rng, 8, 39) if kind == "box" else _log(rng, 8, 20)
        return {"family": family, "kind": kind, "grid": g,
                "rows": max(1, g * g // rng.randint(14, 20)) if kind == "box" else max(1, round(0.4 * g * g))}
    kind = rng.choice(["train", "predict"])
    out = _log(rng, 50, 4000)
    batch = _log(rng, 8, 128)
    return {"family": family, "kind": kind, "hidden": _log(rng, 64, 1024), "out": out,
            "samples": batch * rng.randint(2, 8) if kind == "train" else _log(rng, 1, 512), "batch": batch}


# ---------------------------------------------------------------------------
# the analysed handle of a pattern
# ---------------------------------------------------------------------------
def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


def _settings(s, case):
    s.reg_diag = 1e-9
    s.precision = PRECISION[case["precision"]]
    if case.get("refine", "target") == "target":
        s.target_bwd_err = 1e-10
        s.max_refine_rounds = 20
    if s.symbolic_analysis() != 1:
        raise RuntimeError("symbolic analysis failed")
    return s


def _coupling(n, Ap, Ai, nh):
    """Positions of A's entries in the lower CSC of [H A'; A 0]."""
    col = np.repeat(np.arange(n), np.diff(Ap))
    return np.flatnonzero((col < nh) & (Ai >= nh))


class _System:
    """One analysed system: pattern, base values and the entries that a new seed draws."""

    def __init__(self, case):
        if case["family"] == "indef":
            self.n, self.Ap, self.Ai, self.Ax, _ = P.block_indefinite(case["blocks"], case["size"], seed=1)
            self.free = np.flatnonzero(self.Ax != 0.0)
            self.factor = None
        else:
            self.n, self.Ap, self.Ai, self.Ax, _ = P.kkt_config(case["grid"], case["rows"], case["nnz"], seed=1)
            self.free = _coupling(self.n, self.Ap, self.Ai, case["grid"] ** 3)
        self.s = _settings(lbl.SolverSettings(self.n, self.Ap, self.Ai, self.Ax), case)

    def values(self, rng):
        Ax = self.Ax.copy()
        Ax[self.free] = rng.standard_normal(len(self.free))
        return Ax


class _Batch:
    def __init__(self, case):
        rng = np.random.default_rng(1)
        blocks, self.parts, at, row = [], [], 0, 0
        for _ in range(case["count"]):
            r, c = (int(v) for v in rng.integers(case["lo"], case["hi"] + 1, size=2))
            m = int(rng.integers(1, case["rows"] + 1))
            A = P.random_rows(rng, m, r * c, 4)
            n, Ap, Ai, Ax = P.lower_csc(P.kkt(P.laplacian_2d(r, c, 1e-2), A))
            blocks.append((n, Ap, Ai, Ax))
            self.parts.append((row, n, at, _coupling(n, Ap, Ai, r * c) + at))
            at += len(Ax)
            row += n
        self.blocks = blocks
        self.Ax = np.concatenate([b[3] for b in blocks])
        self.free = np.concatenate([p[3] for p in self.parts])
        self.s = _settings(lbl.BatchSolverSettings(blocks), case)
        self.n = self.s.n

    def values(self, rng):
        Ax = self.Ax.copy()
        Ax[self.free] = rng.standard_normal(len(self.free))
        return Ax


class _Qp:
    def __init__(self, case):
        if case["kind"] == "box":
            self.H, _, self.A, _, self.C, self.d = P.qp_config(grid=case["grid"], meq=case["rows"], seed=1)
            self.s = qp.Nasoq(self.H, np.zeros(self.H.shape[0]), self.A, np.zeros(self.A.shape[0]), self.C, self.d)
            self.s.eps_abs = 1e-8
            self.s.variant = qp.FIXED
        else:
            self.family = learned.ParametricQpFamily(grid=case["grid"], ineq_ratio=case["rows"] / case["grid"] ** 2,
                                                     seed=1)
            self.H, self.A, self.C, self.d = self.family.H, None, self.family.B, self.family.d
            self.s = self.family.solver()

    def linear(self, case, seed):
        rng = np.random.default_rng(seed)
        if case["kind"] == "box":
            # right-hand sides that a point of the box attains
            return (rng.standard_normal(self.H.shape[0]), self.A @ rng.uniform(-0.4, 1.0, self.H.shape[0]))
        return self.family.q(self.family.thetas(1, seed)[0]), None


@functools.lru_cache(maxsize=2)
def _plan(key):
    case = dict(key)
    if case["family"] == "batch":
        return _Batch(case)
    if case["family"] == "qp":
        return _Qp(case)
    p = _System(case)
    if case["family"] == "solve":  # the matrix of this family is fixed: its factor is what the program keeps
        p.Ax = p.values(np.random.default_rng(2))
        p.factored = False
    return p


def _mlp_inputs(case, seed):
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((case["samples"], 32)).astype(np.float32)
    W = rng.standard_normal((32, case["out"])) / math.sqrt(32)
    Y = (X @ W > 0.7).astype(np.float32)
    return X, Y


def prepare(case, seed):
    if case["family"] == "mlp":
        X, Y = _mlp_inputs(case, seed)
        net = learned.ActiveSetPredictor(32, case["out"], hidden=(case["hidden"], case["hidden"]), seed=seed,
                                         max_batch=case["batch"])
        return {"case": case, "net": net, "X": X, "Y": Y}
    p = _plan(_key(case))
    if case["family"] == "qp":
        q, a = p.linear(case, seed)
        return {"case": case, "s": p.s, "q": q, "a": a}
    rng = np.random.default_rng(seed)
    if case["family"] == "solve":
        if not p.factored:
            p.s.set_values(p.Ax)
            p.s.numerical_factorization()
            p.factored = True
        return {"case": case, "s": p.s, "B": rng.uniform(-1.0, 1.0, (p.n, case["nrhs"]))}
    Ax = p.values(rng)
    return {"case": case, "s": p.s, "Ax": Ax, "B": rng.uniform(-1.0, 1.0, (p.n, case.get("nrhs", 1)))}


def run(state):
    case = state["case"]
    if case["family"] == "mlp":
        net = state["net"]
        if case["kind"] == "predict":
            return net.predict_raw(state["X"])
        loss = net.train_raw(state["X"], state["Y"], case["batch"], 1, 1e-3, seed=3)
        return {"loss": float(loss), "params": net.params()}
    s = state["s"]
    if case["family"] == "qp":
        s.set_linear(q=state["q"], a=state["a"])
        status = s.solve()
        return {"status": int(status), "x": s.primal_vars.copy(), "z": s.dual_vars.copy(),
                "y": s.dual_vars_eq.copy()}
    if case["family"] != "solve":
        s.set_values(state["Ax"])
        s.numerical_factorization()
    return s.solve_only(state["B"])


def work(case):
    """Bytes: K and the right-hand sides read, the factor written once and read
    by each direction of the sweep, the solution written.  Flops: sum of the
    squared column counts of L for the factorization, four per entry of L and
    right-hand side for a solve.  A QP repeats the solve for every active-set
    iteration (about 0.07 n with box rows, 0.1 n with coupled ones) and
    updates a small part of the factor."""
    if case["family"] == "mlp":
        h, o, s = case["hidden"], case["out"], case["samples"]
        weights = 32 * h + h + h * h + h + h * o + o
        io = 4.0 * s * (32 + o)
        if case["kind"] == "predict":
            return {"bytes": io + 2.0 * weights, "flops": 2.0 * s * weights}
        steps = s // case["batch"]
        # a step reads and writes the parameters and both Adam moments
        return {"bytes": io + 24.0 * weights * steps, "flops": 6.0 * steps * case["batch"] * weights}
    p = _plan(_key(case))
    size = 8.0 if case.get("precision", "f64") == "f64" else 4.0
    if case["family"] == "qp":
        n = case["grid"] ** 2
        nnz = p.H.nnz + p.C.nnz + (p.A.nnz if p.A is not None else 0)
        iters = max(1.0, (0.07 if case["kind"] == "box" else 0.1) * n)
        lnz = 4.0 * n * math.log2(max(n, 2))  # a nested-dissection factor of a 2-D mesh
        return {"bytes": iters * (2 * 8.0 * lnz + 12.0 * nnz + 16.0 * n), "flops": iters * 4.0 * lnz}
    fl, lnz = p.s.flops()
    n, nrhs = p.n, case.get("nrhs", 1)
    sweeps = 2 * size * lnz + 16.0 * n * nrhs
    if case["family"] == "solve":
        return {"bytes": sweeps, "flops": 4.0 * lnz * nrhs}
    return {"bytes": 12.0 * len(p.Ax) + size * lnz + sweeps, "flops": fl + 4.0 * lnz * nrhs}


def tolerance(case):
    if case["family"] == "mlp":
        # BF16 products; Adam moves a weight whose gradient is rounding noise by its learning rate either way
        return {"rel": 1e-3, "max": 0.5}
    if case["family"] in ("qp", "indef"):
        return {"rel": 1e-9}
    if case.get("refine", "target") == "target":
        # refined to a backward error of 1e-10: two factorizations whose atomic
        # sums came in another order differ by 1e-8 (2-norm), 4e-6 (largest)
        return {"rel": 2e-7, "max": 1e-4}
    return {"rel": 1e-10, "max": 1e-8}


# ---------------------------------------------------------------------------
# 64-bit references
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _dense_solve(n, Ap, Ai, Ax, B):
    dev = _device()
    K = torch.zeros((n, n), dtype=torch.float64, device=dev)
    col = torch.from_numpy(np.repeat(np.arange(n), np.diff(Ap))).to(dev)
    row = torch.from_numpy(Ai.astype(np.int64)).to(dev)
    v = torch.from_numpy(Ax).to(dev)
    K[row, col] = v
    K[col, row] = v
    b = torch.from_numpy(np.ascontiguousarray(B)).to(dev)
    LU, piv = torch.linalg.lu_factor(K)
    x = torch.linalg.lu_solve(LU, piv, b)
    for _ in range(2):
        x = x + torch.linalg.lu_solve(LU, piv, b - K @ x)
    return x.cpu().numpy()


def _dense_qp(H, q, A, a, C, d):
    """Primal-dual interior point on dense matrices, then one solve of the KKT
    systems of the active sets it ends at: (x, z, y)."""
    dev = _device()
    t = lambda v: torch.from_numpy(np.ascontiguousarray(v, dtype=np.float64)).to(dev)
    H, q, C, d = t(H.toarray()), t(q), t(C.toarray()), t(d)
    n, mi = H.shape[0], C.shape[0]
    A = t(A.toarray()) if A is not None else torch.zeros((0, n), dtype=torch.float64, device=dev)
    a = t(a) if a is not None else torch.zeros(0, dtype=torch.float64, device=dev)
    me = A.shape[0]
    zero = torch.zeros((me, me), dtype=torch.float64, device=dev)
    x, y = torch.zeros_like(q), torch.zeros_like(a)
    s, z = torch.ones_like(d), torch.ones_like(d)
    for _ in range(80):
        rd = H @ x + q + A.T @ y + C.T @ z
        rp, rc = A @ x - a, C @ x + s - d
        mu = torch.dot(s, z) / mi
        if max(float(rd.abs().max()), float(rc.abs().max()), float(mu)) < 1e-11:
            break
        M = torch.cat([torch.cat([H + C.T @ ((z / s)[:, None] * C), A.T], 1), torch.cat([A, zero], 1)], 0)
        LU, piv = torch.linalg.lu_factor(M)

        def step(target, corr):
            rs = s * z + corr - target
            g = -(rd + C.T @ ((z * rc - rs) / s))
            u = torch.linalg.lu_solve(LU, piv, torch.cat([g, -rp])[:, None])[:, 0]
            ds = -rc - C @ u[:n]
            return u[:n], u[n:], ds, (-rs - z * ds) / s

        def longest(v, dv):
            r = torch.where(dv < 0, -v / dv, torch.full_like(v, float("inf")))
            return min(1.0, 0.995 * float(r.min()))

        dx, dy, ds, dz = step(0.0, 0.0)
        al, az = longest(s, ds), longest(z, dz)
        sigma = float(torch.dot(s + al * ds, z + az * dz) / mi / mu) ** 3
        dx, dy, ds, dz = step(sigma * mu, ds * dz)
        al = min(longest(s, ds), longest(z, dz))
        x, y, s, z = x + al * dx, y + al * dy, s + al * ds, z + al * dz
    on = z > s
    for _ in range(20):  # the active set that solve shows to be the optimal one
        act = torch.nonzero(on)[:, 0]
        E = torch.cat([A, C[act]], 0)
        k = E.shape[0]
        M = torch.cat([torch.cat([H, E.T], 1),
                       torch.cat([E, torch.zeros((k, k), dtype=torch.float64, device=dev)], 1)], 0)
        b = torch.cat([-q, a, d[act]])[:, None]
        LU, piv = torch.linalg.lu_factor(M)
        u = torch.linalg.lu_solve(LU, piv, b)
        u = (u + torch.linalg.lu_solve(LU, piv, b - M @ u))[:, 0]
        zf = torch.zeros_like(d)
        zf[act] = u[n + me:]
        right = torch.where(on, zf > 0, C @ u[:n] > d + 1e-12)
        if torch.equal(right, on):
            break
        on = right
    return u[:n].cpu().numpy(), zf.cpu().numpy(), u[n:n + me].cpu().numpy()


def _mlp_forward(par, dims, X):
    i, h, h2, o = dims
    at, out = 0, []
    for rows, cols in ((h, i), (h2, h), (o, h2)):
        W = par[at:at + rows * cols].reshape(rows, cols)
        at += rows * cols
        out.append((W, par[at:at + rows]))
        at += rows
    a = X
    for W, b in out[:2]:
        a = torch.relu(a @ W.T + b)
    return a @ out[2][0].T + out[2][1]


def exact(case, seed):
    if case["family"] == "mlp":
        if case["kind"] == "train":
            return None  # the order of the samples and Adam's state are the library's own
        st = prepare(case, seed)
        par = torch.from_numpy(st["net"].params().astype(np.float64))
        dims = (32, case["hidden"], case["hidden"], case["out"])
        return torch.sigmoid(_mlp_forward(par, dims, torch.from_numpy(st["X"].astype(np.float64)))).numpy()
    if case["family"] == "qp":
        p = _plan(_key(case))
        if p.H.shape[0] + p.C.shape[0] > DENSE:
            return None
        q, a = p.linear(case, seed)
        x, z, y = _dense_qp(p.H, q, p.A, a, p.C, p.d)
        return {"status": None, "x": x, "z": z, "y": y}
    if case["family"] == "batch":
        p = _plan(_key(case))
        if max(part[1] for part in p.parts) > DENSE or sum(part[1] ** 3 for part in p.parts) > 2e12:
            return None
        st = prepare(case, seed)
        out = np.empty((p.n, 1))
        for (row, n, at, _), (_, Ap, Ai, Ax) in zip(p.parts, p.blocks):
            out[row:row + n] = _dense_solve(n, Ap, Ai, st["Ax"][at:at + len(Ax)], st["B"][row:row + n])
        return out
    if case["family"] == "indef":
        n = case["blocks"] * case["size"]
    else:
        n = case["grid"] ** 3 + case["rows"]
    if n > DENSE:
        return None
    p = _plan(_key(case))
    st = prepare(case, seed)
    return _dense_solve(p.n, p.Ap, p.Ai, st.get("Ax", p.Ax), st["B"])
