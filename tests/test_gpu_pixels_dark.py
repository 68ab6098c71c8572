"""Longwave pixels without radiance, or with an error larger than it: rays
that leave the atmosphere, few realisations. Their structs from draw_map are
the host's bit for bit, and making them costs no more than others do."""
import time

import numpy as np
import pytest

from htrdr_kmin_amd import _ffi as F
from htrdr_kmin_amd import atmosphere as A
from htrdr_kmin_amd import hip as H

from test_gpu_pixels import check, lw  # noqa: F401

pytestmark = pytest.mark.gpu


def sky(height, width, rows, wlen, up=1.0):
    pos = (1600.0, 1600.0, height)
    return A.map_preset(0, width=width, height=rows, spp=2, spectral_type=F.SPECTRAL_LW, wlen_range=wlen,
                        ref_temperature=290.0, solver=F.SOLVER_WAVEFRONT_FP32, pos=pos,
                        tgt=(pos[0], pos[1] + 0.2, pos[2] + up))


@pytest.mark.parametrize("wlen", [(4000.0, 20000.0), (9999.0, 10001.0), (10000.0, 10000.0),
                                  (4000.0, 4000.4), (4000.0, 4004.1)])
@pytest.mark.parametrize("height", [1e5, 1.5e4, 5e3])
def test_dark_pixels(lw, wlen, height):  # noqa: F811
    dev = check(lw, sky(height, 53, 29, wlen))
    dark = dev["radiance_E"] == 0
    assert dark.any()
    if height == 1e5:
        assert dark.all() and (dev["temperature_E"] == 200.0 * 2.0 ** -21).all()


def test_a_dark_image_takes_no_longer_than_its_rendering(lw):  # noqa: F811
    """256x256 pixels whose temperatures the host would search one by one take
    390 ms; the rest of such an image, 2 ms."""
    d = sky(1e5, 256, 256, (4000.0, 20000.0))
    times = []
    for _ in range(4):
        H.synchronize()
        t = time.perf_counter()
        dev = lw.draw_map(d)
        times.append(time.perf_counter() - t)
    assert (dev["radiance_E"] == 0).all()
    assert min(times) < 0.06, times
