"""htgx_render_accum_noalloc at sizes where its scratch does not hold the
chunks of the map at once: the same accumulators bit for bit as
htgx_render_accum, which takes them in one launch."""
import numpy as np
import pytest

from htrdr_kmin_amd import _ffi as F
from htrdr_kmin_amd import atmosphere as A

from test_zz_no_alloc import FIELDS, both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,spp,chunk,spectral", [
    (256, 256, 16, 4, F.SPECTRAL_SW),          # 2^20 chunks of one
    (256, 256, 20, 4, F.SPECTRAL_SW),
    (512, 288, 15, 4, F.SPECTRAL_SW),          # 15 chunks a pixel, at most 10 in a launch
    (512, 288, 13, 13, F.SPECTRAL_SW),         # ranges that do not divide the chunks
    (512, 512, 14, 16, F.SPECTRAL_SW),         # chunks of 2
    (200, 160, 12, 4, F.SPECTRAL_SW_CIE_XYZ),
    (512, 480, 7, 7, F.SPECTRAL_SW_CIE_XYZ),   # the planes together, a range at a time
    (800, 672, 7, 7, F.SPECTRAL_SW_CIE_XYZ)])  # plane by plane
def test_noalloc_equals_render_accum_beyond_the_scratch(width, height, spp, chunk, spectral):
    s = A.Synth(0, seed=2)
    kw = {"wlen_range": (500.0, 600.0)} if spectral == F.SPECTRAL_SW_CIE_XYZ else {}
    d = A.map_preset(0, width=width, height=height, spp=spp, spp_offset=3, spectral_type=spectral,
                     solver=F.SOLVER_WAVEFRONT_FP32, **kw)
    with A.Context(s.scene_ptr) as ctx:
        ctx.set_wavefront_params(chunk=chunk)
        r, g = both(ctx, d)
        assert np.all(r["n"] == spp)
        for f in FIELDS:
            assert np.array_equal(r[f], g[f]), f
    s.close()
