"""The pixel structs draw_map makes on the device against those the host makes
of the same accumulators (htgx_finalize_pixels): equal bit for bit, the
brightness temperatures included."""
import numpy as np
import pytest

from htrdr_kmin_amd import _ffi as F
from htrdr_kmin_amd import atmosphere as A
from htrdr_kmin_amd import hip as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lw():
    s = A.Synth(2, seed=5, cloud_def=(32, 32, 32), cloud_upper=(3200.0, 3200.0, 4200.0))
    with A.Context(s.scene_ptr) as ctx:
        yield ctx
    s.close()


def check(ctx, d):
    planes = A.accum_planes(d)
    acc = np.zeros(planes * d.width * d.height, A.ACCUM_DTYPE)
    buf = H.DeviceBuffer(acc.nbytes)
    buf.zero()
    ctx.render_accum(d, buf.address)
    H.synchronize()
    host = A.finalize(d, buf.download(acc))
    dev = ctx.draw_map(d)
    for k in host.dtype.names:
        if k not in ("time_sum", "time_sum2"):
            assert np.array_equal(host[k], dev[k]), k
    return dev


@pytest.mark.parametrize("wlen", [(4000.0, 20000.0), (9999.0, 10001.0), (10000.0, 10000.0),
                                  (4000.0, 4000.4)])
@pytest.mark.parametrize("solver", [F.SOLVER_WAVEFRONT_FP32, F.SOLVER_PLAIN_FP64])
def test_longwave_image(lw, wlen, solver):
    d = A.map_preset(0, width=67, height=31, spp=5, spectral_type=F.SPECTRAL_LW, wlen_range=wlen,
                     ref_temperature=290.0, solver=solver, pos=(1600.0, -1000.0, 5000.0),
                     tgt=(1600.0, -999.5, 4999.134))
    dev = check(lw, d)
    assert (dev["temperature_E"] > 0).all()


@pytest.mark.parametrize("kw", [
    dict(width=33, height=9, spp=3),
    dict(width=16, height=17, spp=2, spectral_type=F.SPECTRAL_SW_CIE_XYZ, wlen_range=(500.0, 600.0)),
    dict(width=21, height=40, spp=3, sensor=F.SENSOR_RECTANGLE, rect_size=(3000.0, 3000.0),
         pos=(3200.0, 3200.0, 2000.0), tgt=(3200.0, 3200.0, 2001.0), up=(0.0, 1.0, 0.0))])
def test_shortwave_pixels(ctx0, kw):
    check(ctx0, A.map_preset(0, solver=F.SOLVER_WAVEFRONT_FP32, **kw))
