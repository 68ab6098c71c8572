"""The FP64 solver's persistent kernel at the edges of its launch rules and in
both of its variants (plane ground and grey materials, or everything), against
the same realisations run one thread each by the debug entry: bit for bit."""
import numpy as np
import pytest

from htrdr_kmin_amd import _ffi as F
from htrdr_kmin_amd import atmosphere as A
from htrdr_kmin_amd import hip as H

pytestmark = pytest.mark.gpu


def sums(ctx, d):
    n = d.width * d.height
    buf = H.DeviceBuffer(n * A.ACCUM_DTYPE.itemsize)
    buf.zero()
    ctx.render_accum(d, buf.address)
    H.synchronize()
    return buf.download(np.zeros(n, A.ACCUM_DTYPE))


def check(ctx, d):
    n, spp = d.width * d.height, d.spp
    pix = np.repeat(np.arange(n, dtype=np.uint64), spp)
    real = np.tile(np.arange(d.spp_offset, d.spp_offset + spp, dtype=np.uint64), n)
    w = ctx.realisations(d, pix, real).reshape(n, spp)
    acc = sums(ctx, d)
    fine = np.isfinite(w)
    assert np.array_equal(acc["n"], fine.sum(1)) and np.array_equal(acc["nfail"], (~fine).sum(1))
    if spp == 1:
        assert np.array_equal(acc["sum"], np.where(fine, w, 0.0)[:, 0])
    # compensated sums of FP64 terms >= 0 against plain ones: a few ulp
    w = np.where(fine, w, 0.0)
    np.testing.assert_allclose(acc["sum"] + acc["sum_c"], w.sum(1), rtol=1e-14, atol=0)
    np.testing.assert_allclose(acc["sum2"] + acc["sum2_c"], (w * w).sum(1), rtol=1e-14, atol=0)


@pytest.mark.parametrize("width,height,spp", [
    (1, 1, 1), (1, 1, 7), (9, 8, 3), (64, 1, 5), (57, 41, 1), (129, 65, 3)])
def test_camera_realisations(ctx0, width, height, spp):
    check(ctx0, A.map_preset(0, width=width, height=height, spp=spp, spp_offset=5, seed=3))


@pytest.mark.parametrize("lw", [False, True])
@pytest.mark.parametrize("ground", ["plane", "mesh", "repeat"])
def test_flux_realisations(lw, ground):
    kw = dict(cloud_def=(32, 32, 32), cloud_upper=(3200.0, 3200.0, 4200.0))
    if ground != "plane":
        kw.update(ground_type=F.GROUND_MESH, hf_res=33, hf_octaves=4, hf_relief=2500.0, hf_hurst=0.7)
    s = A.Synth(2 if lw else 0, seed=2, **kw)
    if ground == "repeat":
        s.scene.repeat_clouds = s.scene.repeat_ground = 1
    d = A.map_preset(2 if lw else 4, width=23, height=17, spp=2, seed=1, pos=(1600.0, 1600.0, 2000.0),
                     tgt=(1600.0, 1600.0, 2001.0), rect_size=(3200.0, 3200.0))
    with A.Context(s.scene_ptr) as ctx:
        check(ctx, d)
        assert ground == "plane" or sums(ctx, d)["nfail"].sum() > 0  # samples under the terrain
    s.close()


@pytest.mark.parametrize("kw", [
    dict(spectral_type=F.SPECTRAL_SW, wlen_range=(500.0, 600.0)),
    dict(spectral_type=F.SPECTRAL_SW, wlen_range=(550.0, 550.4)),
    dict(projection=1, ortho_height=4000.0), dict(lens_radius=40.0, focal_dst=5000.0)])
def test_general_variant(ctx0, kw):
    check(ctx0, A.map_preset(0, width=19, height=11, spp=2, seed=4, **kw))
