"""FP32 calls in flight together, whose results are those of the same calls one
at a time, bit for bit (the run times of the realisations aside)."""
import ctypes as C
import threading

import pytest

from htrdr_kmin_amd import _ffi as F
from htrdr_kmin_amd import atmosphere as A
from htrdr_kmin_amd import hip as H

from test_gpu_slices import buffer, one_at_a_time, same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    s = A.Synth(0, seed=5, nbands=4, wlen_lo=380.0, wlen_hi=780.0)
    with A.Context(s.scene_ptr) as c:
        yield c
    s.close()


@pytest.mark.parametrize("spectral", [F.SPECTRAL_SW, F.SPECTRAL_SW_CIE_XYZ])
def test_the_wavelength_range_changes_between_calls(ctx, spectral):
    def band(lo, hi):
        return A.map_preset(0, width=48, height=40, spp=8, seed=3, solver=F.SOLVER_WAVEFRONT_FP32,
                            spectral_type=spectral, wlen_range=(lo, hi))
    ds = [band(500.0, 600.0), band(400.0, 760.0), band(450.0, 550.0)]
    accs, stream = [buffer(d) for d in ds], H.Stream()
    for _ in range(2):
        for d, acc in zip(ds, accs):
            ctx.render_accum(d, acc.address, stream.h.value)
    stream.synchronize()
    stream.destroy()
    for d, acc in zip(ds, accs):
        assert same(acc, one_at_a_time(ctx, [d, d]), d)


@pytest.mark.parametrize("mode", [0, 1])  # global, thread-local: both refuse allocations
@pytest.mark.parametrize("calls,elsewhere", [(1, False), (3, False), (2, True)])
def test_capture_after_calls_on_a_stream(mode, calls, elsewhere):
    """From a new context, calls on a stream, then the capture of one like
    them, on it or on another one, replayed with larger ones in between."""
    h = H.hip()
    s = A.Synth(0, seed=6)
    d, e = (A.map_preset(0, width=w, height=w, spp=8, seed=3, solver=F.SOLVER_WAVEFRONT_FP32)
            for w in (40, 64))
    graph, run = C.c_void_p(), C.c_void_p()
    acc, before, other, stream = buffer(d), buffer(d), buffer(e), H.Stream()
    first = H.Stream() if elsewhere else stream
    with A.Context(s.scene_ptr) as ctx:
        for _ in range(calls):
            ctx.render_accum(d, before.address, first.h.value)
        H.ok("hipStreamBeginCapture", h.hipStreamBeginCapture(stream.h, C.c_int(mode)))
        ctx.render_accum(d, acc.address, stream.h.value)
        H.ok("hipStreamEndCapture", h.hipStreamEndCapture(stream.h, C.byref(graph)))
        H.ok("hipGraphInstantiate", h.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
        for _ in range(3):
            H.ok("hipGraphLaunch", h.hipGraphLaunch(run, stream.h))
            ctx.render_accum(e, other.address, stream.h.value)
        H.ok("hipGraphLaunch", h.hipGraphLaunch(run, stream.h))
        H.synchronize()
        assert same(before, one_at_a_time(ctx, [d] * calls), d)
        assert same(acc, one_at_a_time(ctx, [d] * 4), d)
        assert same(other, one_at_a_time(ctx, [e] * 3), e)
        h.hipGraphExecDestroy(run)
        h.hipGraphDestroy(graph)
        stream.destroy()
    s.close()


def test_calls_of_one_thread_while_another_captures(ctx):
    """Calls in flight of one context while another thread captures, in global
    mode, a call of another one."""
    h = H.hip()
    s = A.Synth(0, seed=7)
    d = A.map_preset(0, width=40, height=40, spp=8, seed=3, solver=F.SOLVER_WAVEFRONT_FP32)
    graph, run = C.c_void_p(), C.c_void_p()
    acc, other = buffer(d), buffer(d)
    streams = [H.Stream(), H.Stream()]
    errors = []

    def calls():
        try:
            for _ in range(3):
                ctx.render_accum(d, other.address, streams[1].h.value)
        except Exception as e:
            errors.append(e)

    with A.Context(s.scene_ptr) as captured:
        captured.render_accum(d, acc.address, streams[0].h.value)
        calls()  # the buffers of calls in flight exist
        H.synchronize()
        H.ok("hipStreamBeginCapture", h.hipStreamBeginCapture(streams[0].h, C.c_int(0)))
        t = threading.Thread(target=calls)
        t.start()
        t.join()
        captured.render_accum(d, acc.address, streams[0].h.value)
        H.ok("hipStreamEndCapture", h.hipStreamEndCapture(streams[0].h, C.byref(graph)))
        H.ok("hipGraphInstantiate", h.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
        for _ in range(3):
            H.ok("hipGraphLaunch", h.hipGraphLaunch(run, streams[0].h))
        H.synchronize()
        assert not errors
        assert same(acc, one_at_a_time(captured, [d] * 4), d)
        assert same(other, one_at_a_time(ctx, [d] * 6), d)
        h.hipGraphExecDestroy(run)
        h.hipGraphDestroy(graph)
        for st in streams:
            st.destroy()
    s.close()


@pytest.mark.parametrize("mode", [0, 1])
def test_calls_on_a_stream_while_one_used_before_is_captured(ctx, mode):
    """Calls of a context leave alone the capture of a stream that it drew on
    before."""
    h = H.hip()
    h.hipMemcpyAsync.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p]
    d = A.map_preset(0, width=40, height=40, spp=8, seed=3, solver=F.SOLVER_WAVEFRONT_FP32)
    graph = C.c_void_p()
    acc, other, copy = buffer(d), buffer(d), buffer(d)
    streams = [H.Stream(), H.Stream()]
    for _ in range(2):  # in flight together: both sets of buffers exist
        ctx.render_accum(d, acc.address, streams[0].h.value)
    H.synchronize()
    H.ok("hipStreamBeginCapture", h.hipStreamBeginCapture(streams[0].h, C.c_int(mode)))
    for _ in range(3):
        ctx.render_accum(d, other.address, streams[1].h.value)
    H.ok("hipMemcpyAsync", h.hipMemcpyAsync(copy.ptr, acc.ptr, acc.nbytes, 3, streams[0].h))
    H.ok("hipStreamEndCapture", h.hipStreamEndCapture(streams[0].h, C.byref(graph)))
    h.hipGraphDestroy(graph)
    H.synchronize()
    assert same(acc, one_at_a_time(ctx, [d] * 2), d)
    assert same(other, one_at_a_time(ctx, [d] * 3), d)
    for st in streams:
        st.destroy()
