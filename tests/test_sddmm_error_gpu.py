"""The error of the product on a block pattern against 80 bits.

At most 1.15 times that of sums by thread, wave and chunk of 512 states, which is how it used to be summed; the figures
of that form, relative, in the Frobenius norm over the pattern, are below.  One chain over a chunk's states and one over
the chunks were 1.4 to 1.6 times as far off."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,t,no,dims,former", [(oh.OMX_F64, np.float64, 250, (5, 5, 5), 1.45e-16),
                                                 (oh.OMX_F64, np.float64, 1458, (4, 4, 4), 1.74e-16),
                                                 (oh.OMX_F64, np.float64, 8192, (3, 3, 3), 2.19e-16),
                                                 (oh.OMX_F32, np.float32, 1458, (4, 4, 4), 1.48e-16),
                                                 (oh.OMX_F32, np.float32, 8192, (3, 3, 3), 1.97e-16)])
def test_error(ctx, dt, t, no, dims, former):
    g = np.random.default_rng(3)
    nb = 4 * int(np.prod(dims))
    cp, ri, bv = oh.lattice_bsr(dims, 0)
    a, b = (g.standard_normal((no, nb)).astype(t) for _ in range(2))
    A, B, D = oh.DMat.from_host(ctx, a, dt), oh.DMat.from_host(ctx, b, dt), oh.Bsr(ctx, nb, cp, ri, np.zeros_like(bv))
    oh.sddmm(ctx, A, B, D)
    on = oh.bsr_to_dense(nb, cp, ri, np.ones_like(bv)) != 0
    ref = (a.astype(np.longdouble).T @ b.astype(np.longdouble))[on]
    err = np.linalg.norm((oh.bsr_to_dense(nb, cp, ri, D.values())[on] - ref).astype(float))
    assert err <= 1.15 * former * np.linalg.norm(ref.astype(float)), err / np.linalg.norm(ref.astype(float)) / former
    for m in (A, B, D):
        m.free()
