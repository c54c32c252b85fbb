"""Device memory of freed matrices is taken again, cleared, safely from several threads, and given back."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu


def _malloc(ctx, n):
    p = C.c_void_p()
    oh.check(oh.lib().omx_malloc(ctx.h, n, C.byref(p)), "omx_malloc")
    return p


def _memory():
    """(free, total) bytes of the device, from the HIP runtime the library is linked with."""
    avail, total = C.c_size_t(), C.c_size_t()
    assert oh.lib().hipMemGetInfo(C.byref(avail), C.byref(total)) == 0
    return avail.value, total.value


def _held(before, limit):
    """Bytes of the device taken since `before`, once the driver has booked the frees (it does so later)."""
    for _ in range(100):
        held = before - _memory()[0]
        if held <= limit:
            break
        time.sleep(0.05)
    return held


def test_block_is_taken_again_and_cleared():
    oh.Ctx(0).close()  # no idle blocks of others
    ctx = oh.Ctx(0)
    for rows, cols in ((7, 3), (1000, 700)):
        a = oh.DMat.from_host(ctx, np.full((rows, cols), 3.0))
        p = a.p.value
        a.free()
        assert oh.lib().omx_free(ctx.h, p) != 0  # free already
        b = oh.DMat(ctx, rows, cols)
        assert b.p.value == p
        assert not b.download().any()
        small = oh.DMat(ctx, rows, max(1, cols // 2))  # b's block is in use, half of it would not do
        assert small.p.value != p
        for m in (small, b):
            m.free()


@pytest.mark.parametrize("count,size", [(100, 1000), (12, 1 << 30)])
def test_pool_is_bounded_and_given_back(count, size):
    ctx, other = oh.Ctx(0), oh.Ctx(0)
    ctx.sync()
    before, total = _memory()
    blocks = [_malloc(ctx, size + 4096 * q) for q in range(count)]
    for p in blocks:
        oh.check(oh.lib().omx_free(other.h, p), "omx_free")  # another context than its own
    limit = total // 64 + (64 << 20)
    assert _held(before, limit) <= limit
    ctx.close()
    assert _held(before, 64 << 20) <= 64 << 20


def test_threads():
    bad = []

    def work(seed):
        ctx = oh.Ctx(0)
        rng = np.random.default_rng(seed)
        for _ in range(40):
            n = int(rng.integers(1, 300))
            m = oh.DMat(ctx, n, n)
            z = m.download()
            m.upload(np.full((n, n), float(seed)))
            k = oh.DMat(ctx, n, n)
            if z.any() or k.download().any() or not (m.download() == seed).all():
                bad.append((seed, n))
            m.free()
            k.free()

    threads = [threading.Thread(target=work, args=(q + 1,)) for q in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
