"""FP32 calls in flight together, whose results are those of the same calls one
at a time, bit for bit (the run times of the realisations aside)."""
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
