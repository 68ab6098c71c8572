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
