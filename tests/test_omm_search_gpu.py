"""The four line-search products in one call: one launch for small results, single products for large ones.

Sizes around the tiles and slices, operands and results with padding rows (NaN in the operands), against numpy
in FP64.  Bound per element: a sum of k products in any order is within (k + 4) unit roundings of the sum of
their magnitudes; the symmetric results are exactly symmetric, where HG D^T is only symmetric to rounding (its
lower triangle is the product's)."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(53)


@pytest.mark.parametrize("dt,prec,t", [(oh.OMX_F64, oh.PREC_F64, np.float64), (oh.OMX_F32, oh.PREC_F32, np.float32)])
@pytest.mark.parametrize("n,k,pad", [(1, 3, 0), (31, 70, 2), (54, 108, 0), (129, 65, 1), (250, 500, 0), (640, 300, 0),
                                     (1458, 200, 3), (2600, 130, 0)])
def test_search_products(ctx, dt, prec, t, n, k, pad):
    X = [rng.standard_normal((n, k)).astype(t) for _ in range(5)]
    d = []
    for a in X:
        m = oh.DMat.from_host(ctx, np.vstack([a, np.full((pad, k), np.nan, t)]), dt)
        m.rows = n
        d.append(m)
    W = [oh.DMat(ctx, n + pad, n, dt) for _ in range(4)]
    for w in W:
        w.rows = n
    oh.omm_search(ctx, *d, *W, prec=prec)
    got = [w.download() for w in W]
    D = X[4].astype(np.float64)
    for q in range(4):
        a = X[q].astype(np.float64)
        ref, mag = a @ D.T, np.abs(a) @ np.abs(D).T
        if q >= 2:
            assert np.array_equal(got[q], got[q].T)
            ref, mag = (np.tril(z) + np.tril(z, -1).T for z in (ref, mag))
        assert np.all(np.abs(got[q] - ref) <= (k + 4) * np.finfo(t).eps * mag), (q, n, k)
    for m in d + W:
        m.free()
