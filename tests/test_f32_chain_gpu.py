"""FP32 products: where the sums over K are carried and where they are one chain.

Results of two 128 tiles per CU and more (2 x 256 tiles) are summed in one FP32 chain over K, smaller ones with
a sum carried every 128 values (or in parts of K).  The mixed solve's stop goes by the rounding of the large
ones, so it is part of the result.  Here the first term is 2^24 and the others are 1/4, so that a chain never
leaves 2^24 (four of them are half a unit, and ties go to even) and a carried sum gets every block but the first
exactly.  Same bits from the symmetric form and from the kernel that stages through registers (tile 0)."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
K = 640


def _operand(ctx, rows, contiguous):
    a = np.full((rows, K), 0.5, np.float32)
    a[:, 0] = 4096.0
    return oh.DMat.from_host(ctx, a.T.copy() if contiguous else a, oh.OMX_F32)


@pytest.mark.parametrize("opA", ["n", "t"])
@pytest.mark.parametrize("opB", ["n", "t"])
@pytest.mark.parametrize("m,n,chain", [(2944, 2816, False), (2945, 2816, True), (2944, 2944, True), (8192, 1024, True),
                                       (8192, 1000, True), (8192, 896, False)])
def test_one_chain_or_carried(ctx, opA, opB, m, n, chain):
    A, B = _operand(ctx, m, opA == "t"), _operand(ctx, n, opB == "n")
    W = oh.DMat(ctx, m, n, oh.OMX_F32)
    for tile in (-1, 0):
        oh.check(oh.lib().omx_gemm_set_tile(ctx.h, tile), "omx_gemm_set_tile")
        oh.gemm(ctx, opA, opB, A, B, W, prec=oh.PREC_F32)
        oh.check(oh.lib().omx_gemm_set_tile(ctx.h, -1), "omx_gemm_set_tile")
        w = W.download()
        if chain:
            assert (w == 2.0 ** 24).all(), tile
        else:  # at least the blocks after the first, in whichever parts of K
            assert (w >= 2.0 ** 24 + 0.25 * (K - 160)).all(), tile
    if m == n and opA == "n" and opB == "t":
        oh.gemm_sym(ctx, A, B, W, prec=oh.PREC_F32)
        assert (W.download() == 2.0 ** 24).all() == chain
    for M in (A, B, W):
        M.free()
