"""The error of the OMM gradient at sizes that the K slice of its pair of products does not divide.

The two products used to be made in separate passes there.  At most 1.15 times the error of that form (relative, in the
Frobenius norm, against 80 bits, FP32 against 64): its figures are below.  One chain over both products was 1.3 to 1.6
times as far off."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
ROWS, COLS = 16, 60
TYPES = {"f32": (oh.OMX_F32, np.float32, np.float64), "f64": (oh.OMX_F64, np.float64, np.longdouble),
         "c128": (oh.OMX_C128, np.complex128, np.clongdouble)}


@pytest.mark.parametrize("dt,n,before", [("f32", 2662, 9.2e-7), ("f64", 2001, 1.42e-15), ("c128", 701, 5.8e-16),
                                         ("c128", 1001, 1.07e-15), ("c128", 2001, 2.05e-15)])
def test_pair(ctx, dt, n, before):
    omx, t, wide = TYPES[dt]
    g = np.random.default_rng(7)

    def rand(*s):
        return (g.standard_normal(s) + (1j * g.standard_normal(s) if t is np.complex128 else 0)).astype(t)

    host = [rand(*s) for s in ((n, 2 * n), (n, 2 * n), (n, n), (n, n))]
    A, B, W1, W2 = (oh.DMat.from_host(ctx, x, omx) for x in host)
    G = oh.DMat(ctx, n, 2 * n, omx)
    oh.omm_calc_G(ctx, W1, W2, A, B, G, prec=oh.PREC_F32 if dt == "f32" else oh.PREC_F64)
    got = G.download()[:ROWS, :COLS].astype(wide)
    a, b, w1, w2 = (x.astype(wide) for x in (host[0][:, :COLS], host[1][:, :COLS], host[2][:ROWS], host[3][:ROWS]))
    ref = 4 * a[:ROWS] - 2 * w2 @ a - 2 * w1 @ b
    assert np.linalg.norm((got - ref).astype(complex)) <= 1.15 * before * np.linalg.norm(ref.astype(complex))
    for m in (A, B, W1, W2, G):
        m.free()
