"""BF16 panel products at the edges of their tiles, slices and parts of K, against FP64 products of the
rounded operands.

The operands are rounded to BF16 on the host as the panels are (to nearest, ties to even), so what is left is
the FP32 accumulation: a sum of k exact products in any order is within (k + 8) 2^-23 of the sum of their
magnitudes, plus one rounding of the result."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(5)


def _bf16(a):
    b = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    b = (b + 0x7FFF + ((b >> 16) & 1)) & 0xFFFF0000
    return b.astype(np.uint32).view(np.float32).astype(np.float64)


@pytest.mark.parametrize("opA", ["n", "t"])
@pytest.mark.parametrize("opB", ["n", "t"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (3, 130, 65), (54, 54, 108), (127, 129, 63), (128, 128, 64), (129, 127, 449),
                                   (255, 257, 130), (256, 300, 1025), (700, 650, 333)])
def test_gemm_bf16_edges(ctx, opA, opB, m, n, k):
    A, B = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    C0 = rng.standard_normal((m, n)).astype(np.float32)
    a, b = _bf16(A), _bf16(B)
    ref = -2.0 * (a @ b) + 0.5 * C0
    size = 2.0 * (np.abs(a) @ np.abs(b))
    bound = (k + 8) * 2.0 ** -23 * size + 2.0 ** -23 * (size + np.abs(C0))
    dA = oh.DMat.from_host(ctx, A if opA == "n" else A.T.copy(), oh.OMX_F32)
    dB = oh.DMat.from_host(ctx, B if opB == "n" else B.T.copy(), oh.OMX_F32)
    dC = oh.DMat.from_host(ctx, C0, oh.OMX_F32)
    oh.gemm(ctx, opA, opB, dA, dB, dC, alpha=-2.0, beta=0.5, prec=oh.PREC_BF16)
    got = dC.download().astype(np.float64)
    for M in (dA, dB, dC):
        M.free()
    assert np.all(np.abs(got - ref) <= bound), np.max(np.abs(got - ref) / bound)


@pytest.mark.parametrize("dt", [oh.OMX_F32, oh.OMX_F64])
@pytest.mark.parametrize("n,k", [(65, 70), (300, 333), (1100, 200)])
def test_gemm_sym_bf16_edges(ctx, dt, n, k):
    """The symmetric form's lower triangle is the full product's bit for bit, the upper its mirror."""
    npdt = np.float32 if dt == oh.OMX_F32 else np.float64
    A = rng.standard_normal((n, k)).astype(npdt)
    dA = oh.DMat.from_host(ctx, A, dt)
    full, sym = oh.DMat(ctx, n, n, dt), oh.DMat(ctx, n, n, dt)
    oh.gemm(ctx, "n", "t", dA, dA, full, prec=oh.PREC_BF16)
    oh.gemm_sym(ctx, dA, dA, sym, prec=oh.PREC_BF16)
    f, s = full.download(), sym.download()
    for M in (dA, full, sym):
        M.free()
    assert np.array_equal(np.tril(s), np.tril(f)) and np.array_equal(s, s.T)
