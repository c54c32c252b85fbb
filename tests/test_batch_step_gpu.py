"""One CG step of k-point batches of one, three and eight systems, against numpy.

Cells whose bands of 64 states and groups of 16 columns are no multiples of 8 (the single system's and the
batch's launch maps of the SpMM differ there), and a basis that 4 does not divide.  The first step makes C + x D
with D = 4 HC - 2 SW HC - 2 HW SC and x the minimum of the line search's quartic, so that every column of H's
and S's products with C and with D counts.  The operators are shifted far below zero, where the quartic has one
minimum.

A system's result does not depend on the batch around it: the same bits in a batch of one.  Against numpy the
step agrees to 1e-8 (complex64: 1e-3) of its largest element: sums of up to nb no = 4e5 rounded terms give 1e-13
(4e-5), and the coefficients cancel a few digits; a column that is missing in any product is off by its own size."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
ETA = 10.0


def _systems(dims, cut, nsys):
    """Operators of nsys k-points of the cell, without the last `cut` basis functions: nb, pattern, blocks, dense."""
    nb = 4 * int(np.prod(dims)) - cut
    out = []
    for s in range(nsys):
        phi = (0.13 * s, 0.29 * s, 0.41 * s)
        cp, ri, h = oh.lattice_bsr_k(dims, 0, phi)
        _, _, sv = oh.lattice_bsr_k(dims, 1, phi)
        col = np.repeat(np.arange(len(cp) - 1), np.diff(cp))
        inside = (4 * ri[:, None, None] + np.arange(4)[None, None, :] < nb) & (4 * col[:, None, None] + np.arange(4)[None, :, None] < nb)
        keep = inside.reshape(-1, 16)  # entry (r, c) of a block at r + 4 c
        h, sv = np.where(keep, h - ETA * sv, 0), np.where(keep, sv, 0)
        full = len(cp) * 4 - 4
        out.append((h, sv, oh.bsr_to_dense(full, cp, ri, h)[:nb, :nb], oh.bsr_to_dense(full, cp, ri, sv)[:nb, :nb]))
    return nb, cp, ri, out


def _step(C, H, S):
    HC, SC = C @ H, C @ S
    HW, SW = HC @ C.conj().T, SC @ C.conj().T
    D = 4 * HC - 2 * SW @ HC - 2 * HW @ SC

    HWd, SWd = HC @ D.conj().T, SC @ D.conj().T
    h = [HW, HWd + HWd.conj().T, D @ H @ D.conj().T]  # HW and SW of C + x D, by powers of x
    w = [SW, SWd + SWd.conj().T, D @ S @ D.conj().T]
    q = np.zeros(5)
    for i in range(3):
        q[i] += 2 * np.real(np.trace(h[i]))
        for j in range(3):
            q[i + j] -= np.real(np.sum(w[i] * h[j].T))
    r = np.roots((q * np.arange(5))[:0:-1])
    r = np.sort(np.real(r[np.abs(np.imag(r)) < 1e-9 * np.abs(r).max()]))
    assert q[4] > 0 and len(r) in (1, 3)
    # the minimum downhill from 0
    return C + (r[0] if len(r) == 1 or r[1] >= 0 else r[2]) * D


@pytest.mark.parametrize("dt,t,tol", [(oh.OMX_C128, np.complex128, 1e-8), (oh.OMX_C64, np.complex64, 1e-3)])
@pytest.mark.parametrize("dims,cut,no", [((3, 3, 3), 0, 54), ((4, 4, 3), 0, 96), ((5, 5, 4), 3, 199), ((6, 6, 6), 2, 432),
                                         ((3, 3, 3), 1, 530)])
def test_first_step(ctx, dt, t, tol, dims, cut, no):
    nb, cp, ri, ops = _systems(dims, cut, 8)
    Cs = [(oh.random_c0(no, nb, 11 + s) + 1j * oh.random_c0(no, nb, 31 + s)).astype(t) for s in range(8)]
    alone = {}
    for nsys in (1, 3, 8):
        for first in range(0, 3 if nsys == 1 else 1):
            part = range(first, first + nsys)
            print("CASE", dims, nb, no, t.__name__, list(part), flush=True)
            B = oh.ZBatch(ctx, no, nb, cp, ri, [ops[s][0] for s in part], [ops[s][1] for s in part], dt=dt)
            B.set_c([Cs[s] for s in part])
            B.solve(eta=0.0, cg_tol=0.0, max_steps=1, check_every=1, use_graph=False)
            got = dict(zip(part, B.get_c()))
            B.free()
            for s in part:
                if s in alone:
                    assert np.array_equal(got[s], alone[s]), (nsys, s)
                elif s < 3:
                    C = Cs[s].astype(np.complex128)
                    ref = _step(C, ops[s][2], ops[s][3])
                    err = np.abs(got[s] - ref).max() / np.abs(ref - C).max()
                    assert err <= tol, (nsys, s, err)
                    alone[s] = got[s]
