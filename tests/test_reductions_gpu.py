"""The CG step's reductions below, at and above the 64 workgroups that one launch adds up itself, against numpy.

Each size twice and in alternation, so that a launch finds the counter as the one before left it.  Bound: a sum
of N products in any order is within (N + 8) 2^-52 of the sum of their magnitudes; the coefficients add at most
four such sums, twice each."""
import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(71)


@pytest.mark.parametrize("sizes", [(1, 33), (255, 256), (256, 257), (300, 54)])
def test_coefficients_around_one_launch(ctx, sizes):
    data = {}
    for n in sizes:
        M = [rng.standard_normal((n, n)) for _ in range(6)]
        H, S, Hd, Sd, Hdd, Sdd = M
        f, a = lambda A, B: np.sum(A * B), lambda A, B: np.sum(np.abs(A * B))  # noqa: E731
        tr = np.trace
        ref = [2 * tr(H) - f(H, S), 2 * (2 * tr(Hd) - f(S, Hd) - f(H, Sd)),
               2 * (tr(Hdd) - f(Sd.T, Hd) - f(Sd, Hd)) - f(Hdd, S) - f(H, Sdd), -2 * (f(Hdd, Sd) + f(Sdd, Hd)), -f(Hdd, Sdd)]
        t = lambda A: np.sum(np.abs(np.diag(A)))  # noqa: E731
        mag = [2 * t(H) + a(H, S), 2 * (2 * t(Hd) + a(S, Hd) + a(H, Sd)),
               2 * (t(Hdd) + a(Sd.T, Hd) + a(Sd, Hd)) + a(Hdd, S) + a(H, Sdd), 2 * (a(Hdd, Sd) + a(Sdd, Hd)), a(Hdd, Sdd)]
        data[n] = [oh.DMat.from_host(ctx, m) for m in M], np.array(ref), np.array(mag)
    for n in sizes * 2:
        d, ref, mag = data[n]
        got = oh.omm_coeff(ctx, *d)
        assert np.all(np.abs(got - ref) <= (n * n + 16) * 2.0 ** -52 * mag), n


@pytest.mark.parametrize("dt,t", [(oh.OMX_F64, np.float64), (oh.OMX_C128, np.complex128)])
def test_dots_around_one_launch(ctx, dt, t):
    z = lambda n, m: (rng.standard_normal((n, m)) + (1j * rng.standard_normal((n, m)) if t == np.complex128 else 0)).astype(t)  # noqa: E731
    for n, m in ((1, 1), (128, 128), (127, 130), (128, 128), (300, 700), (1, 1)):
        G, P = z(n, m), z(n, m)
        got = oh.omm_pr_dots(ctx, oh.DMat.from_host(ctx, G, dt), oh.DMat.from_host(ctx, P, dt))
        ref = [np.sum((G.conj() * (G - P)).real), np.sum((P.conj() * P).real)]
        mag = [2 * np.sum(np.abs(G) * np.abs(G - P)), np.sum(np.abs(P) ** 2)]
        assert np.all(np.abs(np.array(got) - ref) <= (2 * n * m + 16) * 2.0 ** -52 * np.array(mag)), (n, m)
