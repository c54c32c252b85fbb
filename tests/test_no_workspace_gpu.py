"""Products whose workspace the device has no room for run without it: K whole instead of in parts, BF16 from the
stored operands instead of panels.

Whole numbers, small enough to be exact in every order, so the result is that of the same product with room.  The
device is filled until less is free than each product asks for (BF16 1.08 GB of panels, FP64 1.7 and complex128 2.0 GB
of parts), with at least 0.5 GB left."""
import ctypes as C

import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
GB = 1 << 30


def _free():
    avail, total = C.c_size_t(), C.c_size_t()
    assert oh.lib().hipMemGetInfo(C.byref(avail), C.byref(total)) == 0
    return avail.value


def _fill():
    """Blocks that leave 0.5 to 0.9 GB."""
    out = []
    for size in (8 * GB, GB, GB // 4):
        while _free() > size + GB // 2:
            p = C.c_void_p()
            if oh.lib().hipMalloc(C.byref(p), C.c_size_t(size)) != 0:
                oh.lib().hipGetLastError()
                break
            out.append(p)
    return out


@pytest.mark.parametrize("dt,prec,t,n,k", [(oh.OMX_F32, oh.PREC_BF16, np.float32, 8193, 32769),
                                           (oh.OMX_F64, oh.PREC_F64, np.float64, 6574, 13148),
                                           (oh.OMX_C128, oh.PREC_F64, np.complex128, 5013, 10026)])
def test_product_without_workspace(dt, prec, t, n, k):
    ctx = oh.Ctx(0)
    base = np.random.default_rng(5).choice([-1, 1], (n, 301)).astype(t)
    A = oh.DMat.from_host(ctx, np.asfortranarray(np.tile(base, (1, k // 301 + 1))[:, :k]), dt)
    W = oh.DMat(ctx, n, n, dt)
    oh.gemm(ctx, "n", "c", A, A, W, prec=prec)
    ref = W.download()
    W.free()
    ctx2 = oh.Ctx(0)  # without a workspace
    W = oh.DMat(ctx2, n, n, dt)
    ctx.close()  # and the first one's given back
    A.ctx = ctx2
    blocks = _fill()
    print("CASE", n, k, t.__name__, "free", _free(), flush=True)
    try:
        assert GB // 4 < _free() < 0.95 * GB
        oh.gemm(ctx2, "n", "c", A, A, W, prec=prec)
        ctx2.sync()
    finally:
        for p in blocks:
            oh.lib().hipFree(p)
    assert np.array_equal(W.download(), ref)
    for M in (A, W):
        M.free()
    ctx2.close()
