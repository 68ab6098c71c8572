"""What the library does around its kernels, on the CPU: the buffers it holds,
the streams it launches on and what it waits for, recorded by a HIP runtime
without a device (hip_recorder.cpp, preloaded into a process of its own)."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C
from htrdr_kmin_amd import _ffi as F
from htrdr_kmin_amd import atmosphere as A

R = C.CDLL(None)
R.recorder_log.restype = R.recorder_live_bytes.restype = C.c_size_t
R.recorder_log.argtypes = [C.c_char_p, C.c_size_t]
R.recorder_fail_above.argtypes = [C.c_size_t]
synth = A.Synth(0, seed=0, nbands=4, wlen_lo=380.0, wlen_hi=780.0)


def log():
    buf = C.create_string_buffer(R.recorder_log(None, 0) + 1)
    R.recorder_log(buf, len(buf))
    return buf.value.decode().splitlines()


def map_of(width, height, spp, solver=F.SOLVER_WAVEFRONT_FP32, **kw):
    return A.map_preset(0, width=width, height=height, spp=spp, solver=solver, **kw)


def first(lines, what):
    return next(i for i, l in enumerate(lines) if l.startswith(what))


def recorded(f, *args):
    R.recorder_clear()
    f(*args)
    return log()


ACCUM = 1 << 40  # only kernels would read it
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    lib = tmp_path_factory.mktemp("recorder") / "recorder.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", str(lib),
                    os.path.join(HERE, "hip_recorder.cpp")], check=True)

    def call(code):
        before = os.environ.get("LD_PRELOAD")
        env = dict(os.environ, LD_PRELOAD=f"{lib}:{before}" if before else str(lib))
        r = subprocess.run([sys.executable, "-c", PRELUDE + code], cwd=ROOT, env=env, timeout=300,
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
        return r.stdout

    return call


@pytest.mark.parametrize("solver", ["F.SOLVER_WAVEFRONT_FP32", "F.SOLVER_PLAIN_FP64"])
def test_partials_after_a_failed_allocation(run, solver):
    """A call that finds no memory for its partial sums is an error; the next
    one, smaller, has partial sums to write to."""
    run(f"""
small, big = map_of(16, 16, 4, {solver}), map_of(256, 256, 32, {solver})
with A.Context(synth.scene_ptr) as ctx:
    ctx.render_accum(small, ACCUM)
    R.recorder_fail_above(1 << 20)
    try:
        ctx.render_accum(big, ACCUM)
        raise SystemExit("no error")
    except F.HtgxError as e:
        assert e.code == F.MEM_ERR
    lines = recorded(ctx.render_accum, small, ACCUM)
    assert any(l.startswith("malloc") for l in lines[:-2]), lines
""")


@pytest.mark.parametrize("spectral", ["F.SPECTRAL_SW", "F.SPECTRAL_SW_CIE_XYZ"])
@pytest.mark.parametrize("at", [1, 2])
def test_wavelength_tables_after_a_failed_allocation(run, spectral, at):
    """A map of another wavelength range whose tables find no memory is an
    error; the next map of the range before has tables to read."""
    run(f"""
def band(lo, hi):
    return map_of(16, 16, 4, spectral_type={spectral}, wlen_range=(lo, hi))

with A.Context(synth.scene_ptr) as ctx:
    ctx.render_accum(band(500.0, 600.0), ACCUM)
    R.recorder_fail_in({at})
    try:
        ctx.render_accum(band(450.0, 700.0), ACCUM)
    except F.HtgxError as e:
        assert e.code == F.MEM_ERR
        lines = recorded(ctx.render_accum, band(500.0, 600.0), ACCUM)
        assert any(l.startswith("malloc") for l in lines[:-2]), lines
    R.recorder_fail_in(0)
""")


@pytest.mark.parametrize("spectral", ["F.SPECTRAL_SW", "F.SPECTRAL_SW_CIE_XYZ"])
def test_wavelength_tables_outlive_the_drawings_that_read_them(run, spectral):
    """A map of another range waits for the drawings in flight, on whichever
    stream they run, before it frees the tables these read."""
    run(f"""
def band(lo, hi):
    return map_of(16, 16, 4, spectral_type={spectral}, wlen_range=(lo, hi))

with A.Context(synth.scene_ptr) as ctx:
    for i in range(3):
        ctx.render_accum(band(500.0, 600.0), ACCUM, 64)
    last = [l.split()[-1] for l in log() if l.startswith("record stream 0x40 ")][-1]
    lines = recorded(ctx.render_accum, band(450.0, 700.0), ACCUM, 64)
    before = lines[:first(lines, "free")]
    assert last in [l.split()[-1] for l in before if l.startswith("sync event")], lines
""")


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("stream", [0, 64])
def test_a_call_is_captured_after_one_like_it(run, mode, stream):
    """After a call on a stream, or on the null stream, one like it can be
    captured. It draws into partial sums that no other call uses and nothing
    frees while the context lives."""
    run(f"""
d, big = map_of(40, 24, 8), map_of(256, 256, 16)
R.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
ctx = A.Context(synth.scene_ptr)
ctx.render_accum(d, ACCUM, {stream})
graphs = set()
for e in (d, d, big):
    R.hipStreamBeginCapture(64, {mode})
    lines = recorded(ctx.render_accum, e, ACCUM, 64)
    R.hipStreamEndCapture(64, C.byref(C.c_void_p()))
    own = {{l.split()[-1] for l in lines if l.startswith("malloc")}}
    assert [l.split()[-1] for l in lines[len(own):]] == ["0x40"] * 3, lines
    graphs |= own
assert len(graphs) == 2
for _ in range(3):
    lines = recorded(ctx.render_accum, big, ACCUM, 64)
    assert not graphs & {{l.split()[-1] for l in lines if l.startswith("free")}}, lines
""")


def test_a_caller_that_waits_uses_one_set_of_partials(run):
    run("""
R.hipStreamSynchronize.argtypes = [C.c_void_p]
with A.Context(synth.scene_ptr) as ctx:
    d = map_of(64, 48, 8)
    ctx.render_accum(d, ACCUM, 64)
    for _ in range(3):
        R.hipStreamSynchronize(64)
        lines = recorded(ctx.render_accum, d, ACCUM, 64)
        assert not any(l.startswith(("malloc", "stream")) for l in lines), lines
    # calls in flight take a second set, and no third one
    held = R.recorder_live_bytes()
    grown, draws = [], set()
    for _ in range(4):
        lines = recorded(ctx.render_accum, d, ACCUM, 64)
        grown.append(R.recorder_live_bytes() - held)
        draws |= {l.split()[-1] for l in lines if "wavefront_kernel" in l}
        assert all(l.endswith("0x40") for l in lines if "merge" in l), lines
    assert 0 < grown[0] == grown[-1], grown
    assert len(draws) == 2 and "0x40" not in draws, draws
""")


def test_calls_on_the_null_stream_and_counted_ones_draw_there(run):
    run("""
with A.Context(synth.scene_ptr) as ctx:
    d = map_of(64, 48, 8)
    ctx.render_accum(d, ACCUM, 64)
    for stream, count in ((0, False), (64, True), (0, True)):
        ctx.set_counting(count)
        lines = recorded(ctx.render_accum, d, ACCUM, stream)
        # after the call in flight, which uses the same partial sums
        assert lines[0].startswith("wait"), lines
        assert {int(l.split()[-1].replace("(nil)", "0"), 16) for l in lines if l.startswith("launch")} == {stream}
""")


def test_tuning_grows_the_partials_once_per_size(run):
    """A trial is timed twice: the first pays for larger partial sums, the
    second does not."""
    run("""
with A.Context(synth.scene_ptr) as ctx:
    lines = recorded(ctx.autotune, map_of(256, 256, 64), 1e9)
    sizes = [int(l.split()[1]) for l in lines if l.startswith("malloc") and int(l.split()[1]) > 1 << 21]
    assert len(sizes) > 2 and len(set(sizes)) == len(sizes), sizes
""")


def test_a_call_with_no_other_in_flight_draws_on_the_callers_stream(run):
    run("""
R.hipStreamSynchronize.argtypes = [C.c_void_p]

def draws_on(ctx, stream):
    lines = recorded(ctx.render_accum, map_of(64, 48, 8), ACCUM, stream)
    draw = [l for l in lines if "wavefront_kernel" in l]
    assert len(draw) == 1
    return draw[0].endswith(hex(stream))

with A.Context(synth.scene_ptr) as a, A.Context(synth.scene_ptr) as b:
    b.wavefront_params()  # its set-up waits for the device
    for k in range(2):
        assert [draws_on(a, 64) for _ in range(4)] == [True, False, False, False]
        assert [draws_on(b, 80) for _ in range(2)] == [True, False]
        for stream in (64, 80):
            R.hipStreamSynchronize(stream)
""")


def test_noalloc_limit(run):
    """2^20 - 4 chunks of the chunk-size parameter, whatever the chunks are."""
    run("""
with A.Context(synth.scene_ptr) as ctx:
    ctx.wavefront_params()
    def call(*size):
        d = map_of(*size)
        return F.load().htgx_render_accum_noalloc(ctx.handle, C.byref(d), C.c_void_p(ACCUM), None)
    assert call(512, 512, 16) == F.BAD_ARG
    assert recorded(call, 504, 512, 16) and call(504, 512, 16) == F.OK
    for spp, launches in ((16, 1), (20, 1), (24, 1), (33, 2)):
        lines = recorded(call, 256, 256, spp)
        assert sum("wavefront_kernel" in l for l in lines) == launches, (spp, lines)
        assert not any(l.startswith(("malloc", "free")) for l in lines)
""")


def test_the_grid_is_the_parameter(run):
    """The launch has the grid that was asked for, on large longwave maps too;
    a third more of them only where the whole device was (the default)."""
    run("""
def blocks(f, *args):
    return [int(l.split()[3]) for l in recorded(f, *args) if "wavefront_" in l]

lw = dict(spectral_type=F.SPECTRAL_LW, wlen_range=(400.0, 700.0), ref_temperature=290.0)
with A.Context(synth.scene_ptr) as ctx, A.Context(synth.scene_ptr) as other:
    d = map_of(512, 512, 16, **lw)
    top = ctx.wavefront_params()["grid_max"]
    assert top == 768
    for grid, want in ((0, 4 * top * 4 // 3), (top, 4 * top * 4 // 3), (top - 1, 4 * top - 4), (576, 2304), (1, 4)):
        for c in (ctx, other):
            c.set_wavefront_params(grid=grid)
        assert blocks(ctx.render_accum, d, ACCUM) == [want], grid
        for items in ([(ctx, d, ACCUM)], [(ctx, d, ACCUM), (other, d, ACCUM)]):
            plan = A.BatchPlan(items, use_graph=False)
            assert blocks(plan.step) == [want], grid
            plan.close()
""")
