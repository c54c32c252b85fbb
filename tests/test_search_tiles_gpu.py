"""The line-search products have the same bits whichever tile is forced and whether the tuner is on.

Sizes that run as one launch and as four, that a single product would split along K or not, in whole and
partial tiles."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(59)


@pytest.mark.parametrize("dt,prec,t", [(oh.OMX_F64, oh.PREC_F64, np.float64), (oh.OMX_F32, oh.PREC_F32, np.float32)])
@pytest.mark.parametrize("n,k", [(54, 108), (128, 256), (250, 500), (432, 864), (640, 1280), (700, 1500), (1458, 2916)])
def test_bits_do_not_depend_on_the_tile(dt, prec, t, n, k):
    ctx = oh.Ctx(0)
    d = [oh.DMat.from_host(ctx, rng.standard_normal((n, k)).astype(t), dt) for _ in range(5)]
    W = [oh.DMat(ctx, n, n, dt) for _ in range(4)]

    def products():
        for w in W:
            w.upload(np.full((n, n), np.nan, t))
        oh.omm_search(ctx, *d, *W, prec=prec)
        return [w.download() for w in W]

    ref = products()
    for tile in range(8):
        oh.check(oh.lib().omx_gemm_set_tile(ctx.h, tile), "omx_gemm_set_tile")
        for q, a in enumerate(products()):
            assert np.array_equal(a, ref[q]), (n, k, "tile", tile, q)
    oh.check(oh.lib().omx_gemm_set_tile(ctx.h, -1), "omx_gemm_set_tile")
    oh.check(oh.lib().omx_autotune(ctx.h, 1), "omx_autotune")
    for _ in range(2):
        for q, a in enumerate(products()):
            assert np.array_equal(a, ref[q]), (n, k, "tuner", q)
    for m in d + W:
        m.free()
    ctx.close()
