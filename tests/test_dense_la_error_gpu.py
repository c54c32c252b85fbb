"""The error of the triangular solves against 80 bits, next to LAPACK's.

Orders of two and three blocks of 256, a factor of condition number about 3: at most 1.4 times as far off (Frobenius norm)
as LAPACK's substitution on the same operands.  Sums over K in one chain were 1.8 and 1.9 times as far off."""
import numpy as np
import pytest
import scipy.linalg as sla

import ommhip as oh

pytestmark = pytest.mark.gpu


def _factor(n):
    g = np.random.default_rng(3)
    Q, _ = np.linalg.qr(g.standard_normal((n, n)))
    A = (Q * np.logspace(0, -1, n)) @ Q.T
    return np.linalg.cholesky((A + A.T) / 2).T.copy(), g.standard_normal((n, n))


def _solve80(U, B):
    """U^-1 B by substitution in long double."""
    X, U = B.astype(np.longdouble), U.astype(np.longdouble)
    for k in range(len(U) - 1, -1, -1):
        X[k] /= U[k, k]
        X[:k] -= np.outer(U[:k, k], X[k])
    return X


@pytest.mark.parametrize("n", [300, 600])
def test_solve_error(ctx, n):
    U, B = _factor(n)
    ref = _solve80(U, B)
    err = lambda X: float(np.linalg.norm((X.astype(np.longdouble) - ref).astype(float)))  # noqa: E731
    lapack = err(sla.solve_triangular(U, B))
    dU = oh.DMat.from_host(ctx, U)
    for side, trans, b in (("l", "n", B), ("r", "t", B.T)):
        d = oh.DMat.from_host(ctx, b)
        oh.check(oh.lib().omx_trsm(ctx.h, oh.OMX_F64, side.encode(), trans.encode(), n, n, 1.0, dU.p, dU.ld, d.p, d.ld),
                 "trsm")
        X = d.download()
        got = err(X if side == "l" else X.T)
        print("CASE", n, side, trans, got, lapack, flush=True)
        assert got <= 1.4 * lapack
        d.free()
    dU.free()
