"""Dense x dense products on a block pattern at the edges of steps, chunks and blocks, against numpy.

Numbers of states around the step (32 FP64, 64 FP32), the 512 chunk and one and two vectors, odd leading
dimensions, a basis that 4 does not divide, block columns of none to twelve blocks, rows past the last state
filled with NaN, and a leading dimension of 2^26.  Bound per entry: a sum of `no` products in FP64 in any
order, alpha and beta applied: (no + 8) unit roundings of the sum of the magnitudes."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(37)


def _pattern(nb):
    nbc = (nb + 3) // 4
    cols = [np.sort(rng.choice(nbc, rng.integers(0, min(nbc, 12) + 1), replace=False)) for _ in range(nbc)]
    cp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    return cp, np.concatenate(cols).astype(np.int32)


def _check(ctx, dt, t, nb, no, pad, alpha, beta):
    cp, ri = _pattern(nb)
    if len(ri) == 0:
        cp, ri = np.append(np.zeros((nb + 3) // 4, np.int32), np.int32(1)), np.zeros(1, np.int32)
    keep = np.arange(4 * ((nb + 3) // 4)) < nb
    jj = np.repeat(np.arange(len(cp) - 1), np.diff(cp))
    ok = np.einsum("lc,lr->lcr", keep.reshape(-1, 4)[jj], keep.reshape(-1, 4)[ri])  # [block][column][row]
    old = rng.standard_normal((len(ri), 4, 4)) * ok
    P = oh.Bsr(ctx, nb, cp, ri, old.reshape(-1, 16))
    M = [rng.standard_normal((no, nb)).astype(t) for _ in range(2)]
    d = []
    for a in M:
        m = oh.DMat(ctx, no + pad, nb, dt)
        if pad < 8:
            m.upload(np.vstack([a, np.full((pad, nb), np.nan, t)]))
            m.rows = no
        else:
            m.rows = no
            m.upload(a)
        d.append(m)
    oh.sddmm(ctx, d[0], d[1], P, alpha=alpha, beta=beta)
    got = P.values().reshape(-1, 4, 4)
    A, B = (np.pad(a.astype(np.float64), ((0, 0), (0, len(keep) - nb))) for a in M)
    G, Ga = A.T @ B, np.abs(A).T @ np.abs(B)
    blk = lambda X: X.reshape(len(keep) // 4, 4, -1, 4)[ri, :, jj, :].transpose(0, 2, 1)  # noqa: E731
    ref, mag = alpha * blk(G) + beta * old, abs(alpha) * blk(Ga) + abs(beta) * np.abs(old)
    for m in d:
        m.free()
    assert np.all(got[~ok] == 0)
    assert np.all(np.abs(got - ref) <= (no + 8) * 2.0 ** -52 * mag), (nb, no, pad)


@pytest.mark.parametrize("dt,t", [(oh.OMX_F64, np.float64), (oh.OMX_F32, np.float32)])
@pytest.mark.parametrize("nb", [5, 203])
@pytest.mark.parametrize("no", [1, 3, 31, 32, 65, 127, 513, 1062, 4129])
def test_sddmm_edges(ctx, dt, t, nb, no):
    _check(ctx, dt, t, nb, no, 0, 1.0, 0.0)
    _check(ctx, dt, t, nb, no, 3, 1.5, -0.5)


def test_sddmm_chunks_of_large_pattern(ctx):
    _check(ctx, oh.OMX_F64, np.float64, 2001, 1062, 1, 2.0, 0.0)  # five waves per CU: chunks of 512


def test_sddmm_large_leading_dimension(ctx):
    _check(ctx, oh.OMX_F32, np.float32, 5, 70, (1 << 26) - 70, 1.0, 0.0)
