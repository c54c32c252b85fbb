"""The error of FP64 and complex128 products of small results against 80 bits.

At most 1.25 times what it was with K split into parts that fill the chip with 128x128 tiles (complex 64x128), which
is how these products used to be summed; the figures of that form, relative, in the Frobenius norm, are below.  One
chain over K was 2.4 to 3.5 times as far off (complex 1.7 to 3.1)."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
ROWS = 24


def _rel(got, ref):
    return float(np.linalg.norm((got - ref).astype(np.complex128)) / np.linalg.norm(ref.astype(np.complex128)))


@pytest.mark.parametrize("n,k,gram,sym,pair", [(250, 500, 3.1e-16, 2.05e-16, 3.26e-16), (700, 1400, 3.49e-16, 2.26e-16, 3.53e-16)])
def test_f64(ctx, n, k, gram, sym, pair):
    g = np.random.default_rng(7)
    a, b, w1, w2 = (g.standard_normal(s) for s in ((n, k), (n, k), (n, n), (n, n)))
    A, B, W1, W2 = (oh.DMat.from_host(ctx, x) for x in (a, b, w1, w2))
    W, G = oh.DMat(ctx, n, n), oh.DMat(ctx, n, k)
    x = lambda m: m.astype(np.longdouble)  # noqa: E731
    oh.gemm(ctx, "n", "t", A, B, W)
    assert _rel(W.download()[:ROWS], x(a[:ROWS]) @ x(b).T) <= 1.25 * gram
    oh.gemm_sym(ctx, A, A, W)
    assert _rel(np.tril(W.download()[-ROWS:], n - ROWS), np.tril(x(a[-ROWS:]) @ x(a).T, n - ROWS)) <= 1.25 * sym
    oh.omm_calc_G(ctx, W1, W2, A, B, G)
    c = slice(0, 200)
    ref = 4 * x(a[:ROWS, c]) - 2 * x(w2[:ROWS]) @ x(a[:, c]) - 2 * x(w1[:ROWS]) @ x(b[:, c])
    assert _rel(G.download()[:ROWS, c], ref) <= 1.25 * pair
    for m in (A, B, W1, W2, W, G):
        m.free()


@pytest.mark.parametrize("n,k,gram,herm", [(250, 500, 2.76e-16, 3.34e-16), (432, 864, 3.07e-16, 4.48e-16), (700, 1400, 5.3e-16, 6.4e-16)])
def test_c128(ctx, n, k, gram, herm):
    g = np.random.default_rng(7)
    a, b = (g.standard_normal((n, k)) + 1j * g.standard_normal((n, k)) for _ in range(2))
    A, B = (oh.DMat.from_host(ctx, m, oh.OMX_C128) for m in (a, b))
    W = oh.DMat(ctx, n, n, oh.OMX_C128)
    x = lambda m: m.astype(np.clongdouble)  # noqa: E731
    oh.gemm(ctx, "n", "c", A, B, W)
    assert _rel(W.download()[:ROWS], x(a[:ROWS]) @ x(b).conj().T) <= 1.25 * gram
    oh.gemm_sym(ctx, A, A, W)
    assert _rel(np.tril(W.download()[-ROWS:], n - ROWS), np.tril(x(a[-ROWS:]) @ x(a).conj().T, n - ROWS)) <= 1.25 * herm
    for m in (A, B, W):
        m.free()
