"""Complex products at the edges of the direct-to-LDS kernel's tiles and slices, against numpy.

Sizes one below, at and one above the 32 and 64 tiles and the slices of K (8 complex128, 16 complex64),
all nine op combinations, padding rows of NaN, and a leading dimension beyond 2^20 (the staged kernel).
Bound per element: a sum of k products in any order, each of four real multiplications and adds, is within
(2 k + 8) unit roundings of twice the sum of the products' magnitudes."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(9)
TYPES = [(oh.OMX_C128, np.complex128, 2.0 ** -52), (oh.OMX_C64, np.complex64, 2.0 ** -23)]


def _c(r, c, t):
    return (rng.standard_normal((r, c)) + 1j * rng.standard_normal((r, c))).astype(t)


def _op(a, o):
    a = a.astype(np.complex128)
    return a if o == "n" else a.T if o == "t" else a.conj().T


def _dev(ctx, a, dt, pad):
    if pad:
        a = np.vstack([a, np.full((pad, a.shape[1]), np.nan, a.dtype)])
    d = oh.DMat.from_host(ctx, a, dt)
    d.rows -= pad
    return d


@pytest.mark.parametrize("dt,t,eps", TYPES)
@pytest.mark.parametrize("opA", ["n", "t", "c"])
@pytest.mark.parametrize("opB", ["n", "t", "c"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (2, 33, 9), (31, 32, 7), (63, 65, 17), (64, 64, 16), (129, 31, 33), (600, 500, 19),
                                   (70, 64, 300)])
def test_zgemm_tile_edges(ctx, dt, t, eps, opA, opB, m, n, k):
    A, B = _c(*((m, k) if opA == "n" else (k, m)), t), _c(*((k, n) if opB == "n" else (n, k)), t)
    C0 = _c(m, n, t)
    a, b = _op(A, opA), _op(B, opB)
    ref = 1.5 * (a @ b) - 0.5 * C0
    bound = (2 * k + 8) * eps * 2 * (1.5 * (np.abs(a) @ np.abs(b)) + 0.5 * np.abs(C0))
    for pad in (0, 1):
        dA, dB, dC = _dev(ctx, A, dt, pad), _dev(ctx, B, dt, pad), oh.DMat.from_host(ctx, C0, dt)
        oh.gemm(ctx, opA, opB, dA, dB, dC, alpha=1.5, beta=-0.5)
        got = dC.download()
        for M in (dA, dB, dC):
            M.free()
        assert np.all(np.abs(got - ref) <= bound), (pad, np.max(np.abs(got - ref) / bound))


@pytest.mark.parametrize("dt,t,eps", TYPES)
@pytest.mark.parametrize("no,nb", [(1, 4), (31, 65), (54, 108), (250, 130), (700, 64)])
def test_zcalc_G_and_herm_edges(ctx, dt, t, eps, no, nb):
    HW, SW, HC, SC = _c(no, no, t), _c(no, no, t), _c(no, nb, t), _c(no, nb, t)
    d = [_dev(ctx, x, dt, 0) for x in (HW, SW, HC, SC)]
    G, W = oh.DMat(ctx, no, nb, dt), oh.DMat(ctx, no, no, dt)
    oh.omm_calc_G(ctx, *d, G)
    oh.gemm_sym(ctx, d[2], d[2], W)
    g, w = G.download(), W.download()
    for M in d + [G, W]:
        M.free()
    HW, SW, HC, SC = (x.astype(np.complex128) for x in (HW, SW, HC, SC))
    size = 4 * np.abs(HC) + 2 * np.abs(SW) @ np.abs(HC) + 2 * np.abs(HW) @ np.abs(SC)
    assert np.all(np.abs(g - (4 * HC - 2 * SW @ HC - 2 * HW @ SC)) <= (4 * no + 16) * eps * 2 * size)
    assert np.all(np.abs(w - HC @ HC.conj().T) <= (2 * nb + 8) * eps * 2 * (np.abs(HC) @ np.abs(HC).T))
    assert np.array_equal(np.triu(w, 1), np.tril(w, -1).conj().T)


@pytest.mark.parametrize("cplx", [False, True])
def test_leading_dimension_beyond_2_20(ctx, cplx):
    """Lane offsets are 32-bit up to a leading dimension of 2^20; past it the staged kernels take over."""
    m, n, k, ld = 40, 5, 3, (1 << 20) + 3
    dt, t = (oh.OMX_C128, np.complex128) if cplx else (oh.OMX_F64, np.float64)
    A, B = (_c(m, k, t), _c(n, k, t)) if cplx else (rng.standard_normal((m, k)), rng.standard_normal((n, k)))
    dA, dB, dC = oh.DMat.from_host(ctx, A, dt, ld=ld), oh.DMat.from_host(ctx, B, dt), oh.DMat(ctx, m, n, dt)
    oh.gemm(ctx, "n", "c", dA, dB, dC)
    got = dC.download()
    for M in (dA, dB, dC):
        M.free()
    assert np.max(np.abs(got - A @ B.conj().T)) <= 1e-13 * k
