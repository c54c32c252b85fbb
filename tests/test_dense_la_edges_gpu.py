"""Dense factorisations at the edges of their blocks (16 inside a diagonal block, 128, pairs of 256, panels of
512), against numpy in FP64.

Orders one below, at and one above the block sizes, leading dimensions with NaN rows below the operands, all
four triangular solves with alpha, the first non-positive pivot at a block's edges.  Bounds: residuals of
backward-stable size, 20 n 2^-52 of the norms involved (the operands are diagonally dominant)."""
import ctypes as C

import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(21)
EPS = 2.0 ** -52
ORDERS = [15, 16, 17, 127, 128, 129, 255, 256, 257, 383, 385, 511, 513, 641]


def _spd(n):
    a = rng.standard_normal((n, n)) / np.sqrt(n)
    return a @ a.T + np.eye(n)


def _dev(ctx, a, pad):
    d = oh.DMat.from_host(ctx, np.vstack([a, np.full((pad, a.shape[1]), np.nan)]))
    d.rows -= pad
    return d


def _potrf(ctx, d, n):
    info = C.c_int(0)
    oh.check(oh.lib().omx_potrf(ctx.h, oh.OMX_F64, n, d.p, d.ld, C.byref(info)), "potrf")
    return info.value


@pytest.mark.parametrize("n", ORDERS)
def test_potrf_sygst_edges(ctx, n):
    S, H = _spd(n), rng.standard_normal((n, n))
    H = H + H.T
    dS, dH = _dev(ctx, S, 3), _dev(ctx, H, 1)
    assert _potrf(ctx, dS, n) == 0
    oh.check(oh.lib().omx_sygst(ctx.h, oh.OMX_F64, n, dH.p, dH.ld, dS.p, dS.ld), "sygst")
    got, red = dS.download(), dH.download()
    U = np.triu(got)
    assert np.array_equal(np.tril(got, -1), np.tril(S, -1))
    assert np.linalg.norm(U.T @ U - S) <= 20 * n * EPS * np.linalg.norm(S)
    assert np.array_equal(red, red.T)
    assert np.linalg.norm(U.T @ red @ U - H) <= 20 * n * EPS * np.linalg.norm(U) ** 2 * np.linalg.norm(red)
    dS.free()
    dH.free()


@pytest.mark.parametrize("side", ["l", "r"])
@pytest.mark.parametrize("trans", ["n", "t"])
@pytest.mark.parametrize("nu", ORDERS)
def test_trsm_edges(ctx, side, trans, nu):
    other = 70
    U = np.triu(rng.standard_normal((nu, nu)) / np.sqrt(nu)) + 3 * np.eye(nu)
    B = rng.standard_normal((nu, other) if side == "l" else (other, nu))
    dU, dB = _dev(ctx, U + np.tril(np.full((nu, nu), 7.0), -1), 2), _dev(ctx, B, 1)  # only the upper triangle counts
    oh.check(oh.lib().omx_trsm(ctx.h, oh.OMX_F64, side.encode(), trans.encode(), *B.shape, -1.5, dU.p, dU.ld, dB.p, dB.ld),
             "trsm")
    X = dB.download()
    opU = U if trans == "n" else U.T
    res = (opU @ X if side == "l" else X @ opU) + 1.5 * B
    assert np.linalg.norm(res) <= 20 * nu * EPS * np.linalg.norm(U) * np.linalg.norm(X)
    dU.free()
    dB.free()


@pytest.mark.parametrize("n,bad", [(20, 1), (20, 16), (20, 17), (200, 128), (200, 129), (600, 513), (600, 600)])
def test_potrf_first_bad_pivot(ctx, n, bad):
    S = _spd(n)
    S[bad - 1, bad - 1] = -1.0
    dS = _dev(ctx, S, 0)
    assert _potrf(ctx, dS, n) == bad
    dS.free()
