"""FP64 products at the edges of the direct-to-LDS kernel's tiles and slices, against numpy.

Sizes one below, at and one above the 32, 64 and 128 tiles and the 16-wide slice of K, one-element and
one-slice products, and shapes that split K; all four op combinations; operands whose leading dimension is
odd and whose padding rows hold NaN (nothing outside the operand may reach the result).  Bound per element:
an FP64 sum of k products, in any order, is within (k + 4) 2^-52 of the sum of the products' magnitudes."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(77)
EPS = 2.0 ** -52


def _padded(ctx, a, pad):
    """Device copy of a with `pad` extra rows of NaN below it (leading dimension rows + pad)."""
    if pad:
        a = np.vstack([a, np.full((pad, a.shape[1]), np.nan)])
    d = oh.DMat.from_host(ctx, a)
    d.rows -= pad
    return d


@pytest.mark.parametrize("opA", ["n", "t"])
@pytest.mark.parametrize("opB", ["n", "t"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 5, 40), (31, 33, 15), (32, 32, 16), (33, 65, 17), (64, 63, 33),
                                   (127, 129, 31), (130, 67, 300), (700, 690, 47), (1500, 1490, 33), (300, 257, 1025)])
def test_gemm_f64_tile_edges(ctx, opA, opB, m, n, k):
    A, B, C0 = rng.standard_normal((m, k)), rng.standard_normal((k, n)), rng.standard_normal((m, n))
    ref = 1.5 * (A @ B) - 0.5 * C0
    bound = (k + 4) * EPS * (1.5 * (np.abs(A) @ np.abs(B)) + 0.5 * np.abs(C0))
    for pad in (0, 3):
        dA = _padded(ctx, A if opA == "n" else A.T.copy(), pad)
        dB = _padded(ctx, B if opB == "n" else B.T.copy(), pad)
        dC = oh.DMat.from_host(ctx, C0)
        oh.gemm(ctx, opA, opB, dA, dB, dC, alpha=1.5, beta=-0.5)
        got = dC.download()
        for M in (dA, dB, dC):
            M.free()
        assert np.all(np.abs(got - ref) <= bound), (pad, np.max(np.abs(got - ref) / bound))


@pytest.mark.parametrize("no,nb", [(1, 4), (31, 60), (54, 108), (129, 257), (250, 500), (1458, 700)])
def test_calc_G_f64_tile_edges(ctx, no, nb):
    """G = 4HC - 2 SW HC - 2 HW SC in one product for orders that are no multiple of the K slice."""
    HC, SC = rng.standard_normal((no, nb)), rng.standard_normal((no, nb))
    HW, SW = rng.standard_normal((no, no)), rng.standard_normal((no, no))
    ref = 4 * HC - 2 * SW @ HC - 2 * HW @ SC
    bound = (2 * no + 8) * EPS * (4 * np.abs(HC) + 2 * np.abs(SW) @ np.abs(HC) + 2 * np.abs(HW) @ np.abs(SC))
    d = [oh.DMat.from_host(ctx, x) for x in (HW, SW, HC, SC)]
    G = oh.DMat(ctx, no, nb)
    oh.omm_calc_G(ctx, *d, G)
    got = G.download()
    for M in d + [G]:
        M.free()
    assert np.all(np.abs(got - ref) <= bound), np.max(np.abs(got - ref) / bound)


@pytest.mark.parametrize("n,k", [(1, 3), (33, 70), (129, 45), (250, 500), (700, 64), (1458, 200)])
def test_gemm_sym_f64_tile_edges(ctx, n, k):
    """The symmetric form writes both triangles: its lower triangle is the full product's bit for bit."""
    C, S = rng.standard_normal((n, k)), rng.standard_normal((k, k))
    HC = C @ (S + S.T)
    dH, dC = oh.DMat.from_host(ctx, HC), oh.DMat.from_host(ctx, C)
    full, sym = oh.DMat(ctx, n, n), oh.DMat(ctx, n, n)
    oh.gemm(ctx, "n", "t", dH, dC, full)
    oh.gemm_sym(ctx, dH, dC, sym)
    f, s = full.download(), sym.download()
    for M in (dH, dC, full, sym):
        M.free()
    assert np.array_equal(np.tril(s), np.tril(f)) and np.array_equal(s, s.T)
    assert np.all(np.abs(s - HC @ C.T) <= 2 * (k + 4) * EPS * (np.abs(HC) @ np.abs(C).T + np.abs(C) @ np.abs(HC).T))
