"""FP32 maps at the edges of the launch rules -- fewer chunks than wavefronts,
fewer than lanes, empty XCD ranges, ragged tiles, several chunk sizes --
against their single realisations: every realisation once, none twice."""
import numpy as np
import pytest

from htrdr_kmin_amd import _ffi as F
from htrdr_kmin_amd import atmosphere as A
from htrdr_kmin_amd import hip as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,spp", [
    (1, 1, 1), (1, 1, 7), (3, 5, 13), (8, 8, 4), (9, 8, 3), (64, 1, 16), (1, 67, 8), (57, 41, 2),
    (129, 65, 12)])
@pytest.mark.parametrize("grid", [0, 1, 3])
def test_map_holds_every_realisation_once(ctx0, width, height, spp, grid):
    d = A.map_preset(0, width=width, height=height, spp=spp, spp_offset=5, seed=3,
                     solver=F.SOLVER_WAVEFRONT_FP32)
    n = width * height
    pix = np.repeat(np.arange(n, dtype=np.uint64), spp)
    real = np.tile(np.arange(5, 5 + spp, dtype=np.uint64), n)
    w = ctx0.realisations(d, pix, real).reshape(n, spp)
    buf = H.DeviceBuffer(n * A.ACCUM_DTYPE.itemsize)
    buf.zero()
    ctx0.set_wavefront_params(grid=grid)
    try:
        ctx0.render_accum(d, buf.address)
        H.synchronize()
    finally:
        ctx0.set_wavefront_params()
    acc = buf.download(np.zeros(n, A.ACCUM_DTYPE))
    assert np.array_equal(acc["n"], np.full(n, spp))
    # sums of at most 16 FP64 terms >= 0 in another order: a few ulp
    np.testing.assert_allclose(acc["sum"] + acc["sum_c"], w.sum(1), rtol=1e-14, atol=0)
    np.testing.assert_allclose(acc["sum2"] + acc["sum2_c"], (w * w).sum(1), rtol=1e-14, atol=0)


@pytest.mark.parametrize("sensor,spp", [
    (F.SENSOR_CAMERA, 191), (F.SENSOR_CAMERA, 192), (F.SENSOR_RECTANGLE, 193)])
def test_longwave_map_at_the_grid_rule(sensor, spp):
    """A longwave map of 16 realisations a lane of 3 wavefronts per SIMD (256
    units of 3 x 4 x 64 lanes: 192 per pixel of 128x128) takes a larger grid:
    as the slices of it, which do not."""
    s = A.Synth(2, seed=5, cloud_def=(32, 32, 32), cloud_upper=(3200.0, 3200.0, 4200.0))
    kw = dict(width=128, height=128, seed=3, solver=F.SOLVER_WAVEFRONT_FP32)
    preset = 2
    if sensor == F.SENSOR_CAMERA:
        preset = 0
        kw.update(spectral_type=F.SPECTRAL_LW, wlen_range=(4000.0, 20000.0), ref_temperature=290.0,
                  pos=(1600.0, -1000.0, 5000.0), tgt=(1600.0, -999.5, 4999.134))
    with A.Context(s.scene_ptr) as ctx:
        accs = []
        for parts in ([spp], [64, 64, spp - 128]):
            buf = H.DeviceBuffer(128 * 128 * A.ACCUM_DTYPE.itemsize)
            buf.zero()
            off = 0
            for n in parts:
                ctx.render_accum(A.map_preset(preset, spp=n, spp_offset=off, **kw), buf.address)
                off += n
            H.synchronize()
            accs.append(buf.download(np.zeros(128 * 128, A.ACCUM_DTYPE)))
    s.close()
    one, cut = accs
    assert np.array_equal(one["n"], np.full(128 * 128, spp))
    assert np.array_equal(cut["n"], one["n"])
    # sums of at most 193 FP64 terms >= 0, compensated, in another order
    for f in ("sum", "sum2"):
        np.testing.assert_allclose(one[f] + one[f + "_c"], cut[f] + cut[f + "_c"], rtol=1e-13, atol=0)


@pytest.mark.parametrize("ny,nz", [(4094, 4096), (4096, 4096), (4098, 4096)])
def test_grid_of_many_rows(ny, nz):
    """At 2^24 rows of the cloud grid the 24-bit index arithmetic ends and the
    kernels with the full one run: every realisation as on its own."""
    s = A.Synth(0, seed=1, cloud_def=(2, ny, nz))
    with A.Context(s.scene_ptr) as ctx:
        d = A.map_preset(0, width=24, height=20, spp=4, seed=3, solver=F.SOLVER_WAVEFRONT_FP32)
        n = d.width * d.height
        pix = np.repeat(np.arange(n, dtype=np.uint64), 4)
        w = ctx.realisations(d, pix, np.tile(np.arange(4, dtype=np.uint64), n)).reshape(n, 4)
        buf = H.DeviceBuffer(n * A.ACCUM_DTYPE.itemsize)
        buf.zero()
        ctx.render_accum(d, buf.address)
        H.synchronize()
        acc = buf.download(np.zeros(n, A.ACCUM_DTYPE))
    s.close()
    assert w.any()
    np.testing.assert_allclose(acc["sum"] + acc["sum_c"], w.sum(1), rtol=1e-14, atol=0)
