"""Contexts and matrices come and go while another stream is being captured into a graph.

As with hipMalloc and hipFree themselves: in a relaxed capture from any thread, in a thread-local one from
another thread.  The captured graph is whole (its fills run on replay), the calls succeed, and a freed block
comes back cleared."""
import ctypes as C
import threading

import numpy as np
import pytest

import ommhip as oh

pytestmark = pytest.mark.gpu
THREAD_LOCAL, RELAXED = 1, 2


def _block(ctx):
    p = C.c_void_p()
    assert oh.lib().omx_malloc(ctx.h, 1 << 20, C.byref(p)) == 0
    return p


def _calls(ctx, held, out):
    h = C.c_void_p()
    out.append(oh.lib().omx_free(ctx.h, held))
    out.append(oh.lib().omx_malloc(ctx.h, 1 << 20, C.byref(h)))
    out.append(oh.lib().omx_free(ctx.h, h))
    new = C.c_void_p()
    out.append(oh.lib().omx_init(0, C.byref(new)))
    out.append(oh.lib().omx_finalize(new))


@pytest.mark.parametrize("mode,other_thread", [(RELAXED, False), (RELAXED, True), (THREAD_LOCAL, True)])
def test_calls_during_capture(mode, other_thread):
    L = oh.lib()
    ctx, captured = oh.Ctx(0), oh.Ctx(0)
    held = _block(ctx)
    a = oh.DMat.from_host(captured, np.full((300, 50), 2.0))
    b = oh.DMat.from_host(captured, np.full((300, 50), 3.0))
    stream, graph, run = C.c_void_p(L.omx_stream(captured.h)), C.c_void_p(), C.c_void_p()
    captured.sync()
    ctx.sync()
    out = []
    assert L.hipStreamBeginCapture(stream, mode) == 0
    rc = L.omx_zero(captured.h, a.p, 300 * 50 * 8)
    if other_thread:
        t = threading.Thread(target=_calls, args=(ctx, held, out))
        t.start()
        t.join()
    else:
        _calls(ctx, held, out)
    rc = rc or L.omx_zero(captured.h, b.p, 300 * 50 * 8)
    end = L.hipStreamEndCapture(stream, C.byref(graph))
    L.hipGetLastError()
    assert out == [0] * 5 and rc == 0 and end == 0
    assert (a.download() == 2.0).all() and (b.download() == 3.0).all()  # captured, not run
    assert L.hipGraphInstantiate(C.byref(run), graph, None, None, 0) == 0
    for _ in range(3):
        for m in (a, b):
            m.upload(np.full((300, 50), 5.0))
        assert L.hipGraphLaunch(run, stream) == 0
        captured.sync()
        assert not a.download().any() and not b.download().any()
    L.hipGraphExecDestroy(run)
    L.hipGraphDestroy(graph)
    for m in (a, b):
        m.free()
    ctx.close()
    captured.close()
