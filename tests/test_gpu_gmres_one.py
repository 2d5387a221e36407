"""GMRES vector steps of short vectors in one workgroup: refinement of an FP32
factor's solutions, over numbers of right-hand sides and restart lengths."""
import numpy as np
import pytest

from nasoq_amd import lbl
from nasoq_amd import problems as P

pytestmark = pytest.mark.gpu


def gmres(K, M, x, b, mr, cycles):
    """GMRES(mr) on M K x = M b in dense 64-bit arithmetic."""
    for _ in range(cycles):
        r = M @ (b - K @ x)
        rho = np.linalg.norm(r)
        if rho < 1e-15:
            return x
        V, H = [r / rho], np.zeros((mr + 1, mr))
        for k in range(mr):
            w = M @ (K @ V[k])
            for _ in range(2):
                for j, v in enumerate(V):
                    h = v @ w
                    H[j, k] += h
                    w = w - h * v
            H[k + 1, k] = np.linalg.norm(w)
            V.append(w / H[k + 1, k])
        e = np.zeros(mr + 1)
        e[0] = rho
        x = x + np.array(V[:mr]).T @ np.linalg.lstsq(H, e, rcond=None)[0]
    return x


@pytest.mark.parametrize("nrhs", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("mr,cycles", [(1, 1), (2, 2), (3, 1), (17, 1)])  # 17: state beyond the LDS copy
def test_refinement_matches_dense_gmres(nrhs, mr, cycles):
    n, Ap, Ai, Ax, B = P.kkt_config(6, 20, 6, seed=mr, nrhs=nrhs)
    print(f"case gmres nrhs={nrhs} mr={mr} cycles={cycles}", flush=True)
    K = P.lower_to_full(n, Ap, Ai, Ax).toarray()
    s = lbl.SolverSettings(n, Ap, Ai, Ax)
    s.reg_diag, s.precision = 1e-9, lbl.F32
    s.max_inner_iter, s.req_ref_iter = mr, cycles
    assert s.symbolic_analysis() == 1
    s.numerical_factorization()
    X = s.solve_only(B)
    s.req_ref_iter = 0  # the sweeps alone: the first solution, and M^-1 column by column
    X0 = s.solve_only(B)
    M = np.hstack([s.solve_only(np.eye(n)[:, c:c + 8]) for c in range(0, n, 8)])
    for c in range(nrhs):
        ref = gmres(K, M, X0[:, c], B[:, c], mr, cycles)
        # the device applies M in FP32 sweeps: n u32 = 1.4e-5 of a correction a
        # step, over at most 17 steps, with a margin of four
        bound = 1e-3 * np.linalg.norm(ref - X0[:, c]) + 1e-13 * np.linalg.norm(ref)
        assert np.linalg.norm(X[:, c] - ref) <= bound, c
    s.close()


@pytest.mark.parametrize("target", [0.0, 1e-13])
def test_columns_agree_across_the_limit(target):
    # 4352 rows: three columns' steps take one workgroup, four columns' take
    # launches; every column is its own iteration, so each agrees with the
    # column solved alone
    n, Ap, Ai, Ax, B = P.kkt_config(16, 256, 8, seed=3, nrhs=4)
    assert 3 * n <= 1 << 14 < 4 * n
    s = lbl.SolverSettings(n, Ap, Ai, Ax)
    s.reg_diag, s.precision, s.target_bwd_err = 1e-9, lbl.F32, target
    s.max_inner_iter, s.req_ref_iter = 3, 2
    assert s.symbolic_analysis() == 1
    s.numerical_factorization()
    for nrhs in (3, 4):
        print(f"case gmres limit nrhs={nrhs} target={target}", flush=True)
        X = s.solve_only(B[:, :nrhs])
        for c in range(nrhs):
            x = s.solve_only(B[:, c])
            # backward errors of at most 1e-13 each and a condition number of
            # 400 (1-norm): a forward difference of at most 8e-11, in the
            # 2-norm with a margin of ten
            assert np.linalg.norm(X[:, c] - x) <= 1e-9 * np.linalg.norm(x), c
            assert s.backward_error(B[:, c], X[:, c]) <= 1e-13, c
    s.close()
