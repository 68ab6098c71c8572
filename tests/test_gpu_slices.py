"""FP32 calls in flight together -- slices of one map, maps of other sizes,
counted calls and the null stream in between, two streams, a captured call
replayed among others -- against the same calls one at a time: the same
accumulators bit for bit (the run times of the realisations aside)."""
import ctypes as C

import numpy as np
import pytest

from htrdr_kmin_amd import _ffi as F
from htrdr_kmin_amd import atmosphere as A
from htrdr_kmin_amd import hip as H

pytestmark = pytest.mark.gpu

FIELDS = ("sum", "sum_c", "sum2", "sum2_c", "n", "nfail")


def desc(width, height, spp, k, spectral=F.SPECTRAL_SW):
    kw = {"wlen_range": (500.0, 600.0)} if spectral == F.SPECTRAL_SW_CIE_XYZ else {}
    return A.map_preset(0, width=width, height=height, spp=spp, spp_offset=k * spp, seed=3,
                        solver=F.SOLVER_WAVEFRONT_FP32, spectral_type=spectral, **kw)


def planes(d):
    return 3 if d.spectral_type == F.SPECTRAL_SW_CIE_XYZ else 1


def buffer(d):
    b = H.DeviceBuffer(d.width * d.height * planes(d) * A.ACCUM_DTYPE.itemsize)
    b.zero()
    return b


def same(buf, ref, d):
    shape = d.width * d.height * planes(d)
    a, b = (x.download(np.zeros(shape, A.ACCUM_DTYPE)) for x in (buf, ref))
    return all(np.array_equal(a[f], b[f]) for f in FIELDS) and a["n"].all()


def one_at_a_time(ctx, descs):
    ref = buffer(descs[0])
    for d in descs:
        ctx.render_accum(d, ref.address)
        H.synchronize()
    return ref


@pytest.mark.parametrize("width,height,spp,slices,spectral", [
    (1, 1, 1, 5, F.SPECTRAL_SW), (57, 41, 3, 7, F.SPECTRAL_SW), (64, 64, 16, 4, F.SPECTRAL_SW),
    (33, 20, 4, 3, F.SPECTRAL_SW_CIE_XYZ)])
def test_slices_in_flight_equal_slices_one_at_a_time(ctx0, width, height, spp, slices, spectral):
    ds = [desc(width, height, spp, k, spectral) for k in range(slices)]
    acc, stream = buffer(ds[0]), H.Stream()
    for d in ds:
        ctx0.render_accum(d, acc.address, stream.h.value)
    stream.synchronize()
    stream.destroy()
    assert same(acc, one_at_a_time(ctx0, ds), ds[0])


def test_calls_of_other_sizes_and_kinds_in_between(synth0):
    """From a new context: the buffers of the calls grow while others run."""
    shapes = [(8, 8, 2), (64, 48, 8), (9, 7, 4), (96, 96, 8)]
    with A.Context(synth0.scene_ptr) as ctx:
        streams = [H.Stream(), H.Stream()]
        accs = [[buffer(desc(*s, 0)) for s in shapes] for _ in streams]
        for k in range(3):
            for i, s in enumerate(shapes):
                ctx.set_counting(k == 1 and i == 2)
                for st, acc in zip(streams, accs):
                    ctx.render_accum(desc(*s, k), acc[i].address, st.h.value)
                    if k == 1 and i == 2:
                        st.synchronize() # counted calls share their counters
            ctx.set_counting(False)
            null = buffer(desc(16, 16, 4, 0))
            ctx.render_accum(desc(16, 16, 4, 0), null.address)
        H.synchronize()
        assert same(null, one_at_a_time(ctx, [desc(16, 16, 4, 0)]), desc(16, 16, 4, 0))
        for i, s in enumerate(shapes):
            ref = one_at_a_time(ctx, [desc(*s, k) for k in range(3)])
            for acc in accs:
                assert same(acc[i], ref, desc(*s, 0)), s
        for st in streams:
            st.destroy()


def test_captured_call_replayed_among_others(ctx0):
    h = H.hip()
    d, e = desc(40, 24, 8, 0), desc(64, 64, 8, 1)
    graph, run = C.c_void_p(), C.c_void_p()
    acc, other, stream = buffer(d), buffer(e), H.Stream()
    one_at_a_time(ctx0, [d]) # the buffers of a call on its own stream exist
    H.ok("hipStreamBeginCapture", h.hipStreamBeginCapture(stream.h, C.c_int(2)))
    ctx0.render_accum(d, acc.address, stream.h.value)
    H.ok("hipStreamEndCapture", h.hipStreamEndCapture(stream.h, C.byref(graph)))
    H.ok("hipGraphInstantiate", h.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
    for _ in range(3):
        H.ok("hipGraphLaunch", h.hipGraphLaunch(run, stream.h))
        ctx0.render_accum(e, other.address, stream.h.value)
    stream.synchronize()
    assert same(acc, one_at_a_time(ctx0, [d] * 3), d)
    assert same(other, one_at_a_time(ctx0, [e] * 3), e)
    h.hipGraphExecDestroy(run)
    h.hipGraphDestroy(graph)
    stream.destroy()
