"""FP32 products at the edges of the direct-to-LDS kernel's tiles and slices, against numpy in FP64.

Sizes one below, at and one above the 32, 64 and 128 tiles and the 32-wide slice of K, one-element and
one-slice products, and shapes that split K; all four op combinations; operands whose leading dimension is
odd and whose padding rows hold NaN.  Bound per element: an FP32 sum of k products, in any order, rounded to
FP32 after alpha and beta, is within (k + 4) 2^-23 of the sum of the products' magnitudes."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(78)
EPS = 2.0 ** -23


def _f32(*shape):
    return rng.standard_normal(shape).astype(np.float32)


def _dev(ctx, a, pad=0):
    if pad:
        a = np.vstack([a, np.full((pad, a.shape[1]), np.nan, np.float32)])
    d = oh.DMat.from_host(ctx, a, oh.OMX_F32)
    d.rows -= pad
    return d


@pytest.mark.parametrize("opA", ["n", "t"])
@pytest.mark.parametrize("opB", ["n", "t"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 5, 40), (31, 33, 31), (32, 32, 32), (33, 65, 33), (64, 63, 65), (127, 129, 63),
                                   (130, 67, 300), (700, 690, 95), (1500, 1490, 33), (300, 257, 2049)])
def test_gemm_f32_tile_edges(ctx, opA, opB, m, n, k):
    A, B, C0 = _f32(m, k), _f32(k, n), _f32(m, n)
    a, b = A.astype(np.float64), B.astype(np.float64)
    ref = 1.5 * (a @ b) - 0.5 * C0
    bound = (k + 4) * EPS * (1.5 * (np.abs(a) @ np.abs(b)) + 0.5 * np.abs(C0))
    for pad in (0, 3):
        dA = _dev(ctx, A if opA == "n" else A.T.copy(), pad)
        dB = _dev(ctx, B if opB == "n" else B.T.copy(), pad)
        dC = _dev(ctx, C0)
        oh.gemm(ctx, opA, opB, dA, dB, dC, alpha=1.5, beta=-0.5, prec=oh.PREC_F32)
        got = dC.download()
        for M in (dA, dB, dC):
            M.free()
        assert np.all(np.abs(got - ref) <= bound), (pad, np.max(np.abs(got - ref) / bound))


@pytest.mark.parametrize("no,nb", [(1, 4), (31, 60), (54, 108), (129, 257), (250, 500), (1458, 700)])
def test_calc_G_f32_tile_edges(ctx, no, nb):
    """G = 4HC - 2 SW HC - 2 HW SC in one product for orders that are no multiple of the K slice."""
    HC, SC, HW, SW = _f32(no, nb), _f32(no, nb), _f32(no, no), _f32(no, no)
    h, s, hw, sw = (x.astype(np.float64) for x in (HC, SC, HW, SW))
    ref = 4 * h - 2 * sw @ h - 2 * hw @ s
    bound = (2 * no + 8) * EPS * (4 * np.abs(h) + 2 * np.abs(sw) @ np.abs(h) + 2 * np.abs(hw) @ np.abs(s))
    d = [_dev(ctx, x) for x in (HW, SW, HC, SC)]
    G = oh.DMat(ctx, no, nb, oh.OMX_F32)
    oh.omm_calc_G(ctx, *d, G, prec=oh.PREC_F32)
    got = G.download()
    for M in d + [G]:
        M.free()
    assert np.all(np.abs(got - ref) <= bound), np.max(np.abs(got - ref) / bound)


@pytest.mark.parametrize("n,k", [(1, 3), (33, 70), (129, 45), (250, 500), (700, 64), (1280, 200), (1458, 200)])
def test_gemm_sym_f32_tile_edges(ctx, n, k):
    """The symmetric form writes both triangles: its lower triangle is the full product's bit for bit."""
    C, HC = _f32(n, k), _f32(n, k)
    dH, dC = _dev(ctx, HC), _dev(ctx, C)
    full, sym = oh.DMat(ctx, n, n, oh.OMX_F32), oh.DMat(ctx, n, n, oh.OMX_F32)
    oh.gemm(ctx, "n", "t", dH, dC, full, prec=oh.PREC_F32)
    oh.gemm_sym(ctx, dH, dC, sym, prec=oh.PREC_F32)
    f, s = full.download(), sym.download()
    for M in (dH, dC, full, sym):
        M.free()
    assert np.array_equal(np.tril(s), np.tril(f)) and np.array_equal(s, s.T)
