"""SpMM at the edges of its vectors, row chunks and blocks, against numpy.

Numbers of states around the vector and the row chunk, odd leading dimensions (so that columns start at
every alignment), chunk counts that 8 does not divide, and a basis that 4 does not divide, on a random
pattern.  Rows past the last state hold NaN in X and must keep their value in Y.  Bound per element: a sum
of w products (complex: four real ones each), the value rounded to the element type, alpha and beta applied:
(2 w + 8) unit roundings of the sum of the magnitudes, twice that for complex."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(31)
TYPES = [(oh.OMX_F64, np.float64), (oh.OMX_F32, np.float32), (oh.OMX_C128, np.complex128), (oh.OMX_C64, np.complex64)]


def _pattern(nb, cplx):
    """A random operator of about 6 blocks per block column (some empty), dense and in blocks."""
    nbc = (nb + 3) // 4
    cols = [np.sort(rng.choice(nbc, rng.integers(0, min(nbc, 12) + 1), replace=False)) for _ in range(nbc)]
    cp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    ri = np.concatenate(cols).astype(np.int32)
    bv = rng.standard_normal((len(ri), 16)) + (1j * rng.standard_normal((len(ri), 16)) if cplx else 0)
    dense = np.zeros((4 * nbc, 4 * nbc), bv.dtype)
    keep = np.zeros((4 * nbc,), bool)
    keep[:nb] = True
    for J in range(nbc):
        for l in range(cp[J], cp[J + 1]):
            b = bv[l].reshape(4, 4).T * np.outer(keep[4 * ri[l]:4 * ri[l] + 4], keep[4 * J:4 * J + 4])
            bv[l] = b.T.reshape(16)
            dense[4 * ri[l]:4 * ri[l] + 4, 4 * J:4 * J + 4] = b
    return cp, ri, bv, dense[:nb, :nb]


def _dev(ctx, a, dt, ld):
    pad = np.full((ld - a.shape[0], a.shape[1]), np.nan, a.dtype)
    d = oh.DMat.from_host(ctx, np.vstack([a, pad]), dt)
    d.rows = a.shape[0]
    return d


@pytest.mark.parametrize("dt,t", TYPES)
@pytest.mark.parametrize("nb", [5, 1999])
@pytest.mark.parametrize("no", [1, 3, 63, 258, 513, 1155])
def test_spmm_edges(ctx, dt, t, nb, no):
    cplx = np.issubdtype(t, np.complexfloating)
    cp, ri, bv, H = _pattern(nb, cplx)
    A = (oh.Bsr.complex if cplx else oh.Bsr)(ctx, nb, cp, ri, bv)
    z = lambda: (rng.standard_normal((no, nb)) + (1j * rng.standard_normal((no, nb)) if cplx else 0)).astype(t)
    X, Y0 = z(), z()
    eps, wide = np.finfo(t).eps, np.complex128 if cplx else np.float64
    w = 4 * int(np.diff(cp).max())
    for beta, padx, pady in ((0.0, 0, 0), (-0.5, 1, 3)):
        dX, dY = _dev(ctx, X, dt, no + padx), _dev(ctx, Y0, dt, no + pady)
        oh.spmm(ctx, dX, A, dY, alpha=1.5, beta=beta)
        got = dY.download()
        dY.rows += pady
        full = dY.download()
        assert np.isnan(full[no:]).all()
        ref = 1.5 * (X.astype(wide) @ H) + beta * Y0
        bound = (2 * w + 8) * eps * (2 if cplx else 1) * (1.5 * (np.abs(X) @ np.abs(H)) + 0.5 * np.abs(Y0))
        assert np.all(np.abs(got - ref) <= bound), (no, nb, beta, np.max(np.abs(got - ref) / bound))
        dX.free()
        dY.free()
