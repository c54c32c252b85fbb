"""The line-search coefficients are summed in a fixed order, bit for bit.

A solve's trajectory hangs on the last bit of these sums, so their order is part of the result: within a thread
by column, within a wave lanes 32 apart first, then 16, 8, 4, 2 and 1, then the waves, and the workgroups' parts
the same way.  With SW all ones and no diagonal in HW and HWd, coefficient 0 is -sum HW and coefficient 1 is
-2 sum HWd (SWd = 0): products by one are exact, so numpy gives the same bits.  One workgroup, 100 (two
launches) and 361 of them (several parts per thread)."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(71)


def _workgroup(v):
    """Sum of 256 threads' values."""
    w = v.reshape(4, 64)
    for off in (32, 16, 8, 4, 2, 1):
        w = w[:, :off] + w[:, off:2 * off]
    s = 0.0
    for x in w[:, 0]:
        s += x
    return s


def _total(W):
    n = len(W)
    tiles = (n + 31) // 32
    P = np.zeros((32 * tiles, 32 * tiles))
    P[:n, :n] = W
    parts = []
    for J in range(tiles):
        for I in range(tiles):
            t = P[32 * I:32 * I + 32, 32 * J:32 * J + 32]
            v = np.zeros((8, 32))
            for c in range(0, 32, 8):  # thread (ty, tx): row tx of columns ty, ty + 8, ...
                v += t[:, c:c + 8].T
            parts.append(_workgroup(v.ravel()))
    parts = np.array(parts + [0.0] * (-len(parts) % 256)).reshape(-1, 256)
    v = np.zeros(256)
    for p in parts:
        v += p
    return _workgroup(v)


@pytest.mark.parametrize("n", [27, 54, 310, 600])
def test_coefficient_sums(ctx, n):
    HW, HWd = (rng.standard_normal((n, n)) * 10.0 ** rng.integers(-3, 4, (n, n)) for _ in range(2))
    np.fill_diagonal(HW, 0.0)
    np.fill_diagonal(HWd, 0.0)
    d = [oh.DMat.from_host(ctx, a) for a in (HW, np.ones((n, n)), HWd, *(np.zeros((n, n)) for _ in range(3)))]
    c = oh.omm_coeff(ctx, *d)
    assert c[0] == -_total(HW) and c[1] == -2.0 * _total(HWd)
    for m in d:
        m.free()
