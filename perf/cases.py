"""The work a user of this library has it do, as cases that can be timed.

A case is one call (or one short program) through the package's public entry
points: an image or a flux map from a scene that is resident on the GPU, a
progressive render into resident accumulators, a batch of scenes stepped by a
plan, or a one-shot render that also sets the scene up. Scenes are the seeded
synthetic ones of the library's own configurations: 0 the small cloud field,
1 the shortwave image, 2 the longwave map of 8 bands x 16 k-points, 4 the
shortwave flux map over a fractal terrain; the sizes are those of these
configurations, of the tests and of the benchmark, cut to fit a pass of well
under 2 s.

What a pass returns are the map's estimates and its realisation counts. The
pixel structs also hold the time each realisation took; that is a measurement
of the run, not a result, and is left out.

Fields of a case:
  kind     "draw": Context.draw_map; "progressive": slices of realisations
           accumulated on the GPU, then fetched; "batch": a plan over several
           scenes, one step; "oneshot": context, map, close
  preset   configuration of the scene and the map (0, 1, 2 or 4)
  sensor   "camera" or "rectangle" (a flux map)
  spectrum "sw" (550 nm), "sw_band" (discrete 1-nm sampling), "cie", "lw"
  solver   "fp32" (the wavefront solver) or "fp64" (the plain one)
  width, height, spp, slices; nx, ny, nz (cloud cells), nquads, hf_res
  repeat   clouds and terrain repeat along X and Y (options -r and -R)
"""
import math

import numpy as np

from htrdr_kmin_amd import _ffi as F
from htrdr_kmin_amd import atmosphere as A
from htrdr_kmin_amd import hip as H

SOLVERS = {"fp32": F.SOLVER_WAVEFRONT_FP32, "fp64": F.SOLVER_PLAIN_FP64}
# Operations one realisation cannot do without, from the library's own
# counters on the preset scenes (tentative collisions, segments and events per
# realisation) at about 100 operations per collision (one Threefry-2x32 block
# is 75), 60 per segment and 500 per event. Terrain: plus its BVH casts.
OPS = {"sw": 72e3, "lw": 50e3, "terrain": 95e3}


def _case(name, **kw):
    c = {"kind": "draw", "preset": 0, "sensor": "camera", "spectrum": "sw", "solver": "fp32",
         "width": 64, "height": 64, "spp": 32, "slices": 1, "nx": 64, "ny": 64, "nz": 32,
         "nquads": 1, "hf_res": 0, "repeat": False, "scenes": 1}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a look at a scene while its camera is being placed: latency counts
        _case("probe_32x24", width=32, height=24, spp=4),
        # the small configuration as it stands
        _case("image_64", width=64, height=64, spp=32),
        # an image of no round size, a prime number of realisations, 4 k-points
        _case("image_ragged", preset=1, width=253, height=187, spp=13, nx=130, ny=98, nz=54,
              nquads=4),
        # the shortwave image, two slices of a progressive render
        _case("image_1024", kind="progressive", preset=1, width=1024, height=1024, spp=16, slices=2,
              nx=256, ny=256, nz=64),
        # the command line's default image mode: CIE XYZ, 3 channels
        _case("cie_image", spectrum="cie", preset=1, width=256, height=256, spp=16, nx=256, ny=256,
              nz=64),
        # the longwave flux map of the benchmark, 16 of its realisations
        _case("lw_flux_512", preset=2, sensor="rectangle", spectrum="lw", width=512, height=512,
              spp=16, nx=256, ny=256, nz=64, nquads=16),
        # a brightness-temperature image
        _case("lw_image", preset=2, spectrum="lw", width=256, height=256, spp=16, nx=256, ny=256,
              nz=64, nquads=16),
        # the flux map over the 2.1 M-triangle terrain, 4 of its realisations
        _case("terrain_flux_512", preset=4, sensor="rectangle", width=512, height=512, spp=4, nx=512,
              ny=512, nz=128, hf_res=1024),
        # several scenes of uneven sizes in one step of a plan
        _case("batch_uneven", kind="batch", width=64, height=256, spp=64, scenes=8, nx=32, ny=256),
        # the double-precision solver, the default of a map description
        _case("fp64_image", solver="fp64", preset=1, width=128, height=128, spp=32, nx=256, ny=256,
              nz=64),
        _case("fp64_lw_flux", solver="fp64", preset=2, sensor="rectangle", spectrum="lw", width=128,
              height=128, spp=16, nx=256, ny=256, nz=64, nquads=16),
        # a run as the command line makes it: scene set-up, one flux map over
        # a repeated terrain, done
        _case("oneshot_terrain", kind="oneshot", preset=4, sensor="rectangle", width=64, height=64,
              spp=8, nx=256, ny=256, nz=64, hf_res=512, repeat=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: sizes over their logarithm."""
    what = rng.choice(["image", "image", "lw_flux", "lw_image", "cie", "terrain", "batch", "fp64",
                       "oneshot"])
    nx, ny = (2 * _log_int(rng, 16, 128) for _ in range(2))
    nz = 2 * _log_int(rng, 16, 48)
    w, h = _log_int(rng, 16, 640), _log_int(rng, 16, 640)
    spp = _log_int(rng, 1, 64)
    most = {"image": 6000000, "lw_flux": 4000000, "lw_image": 1000000, "cie": 700000,
            "terrain": 500000, "batch": 0, "fp64": 400000, "oneshot": 60000}[what]
    if what == "lw_image":
        w, h = min(w, 256), min(h, 256)
    if what == "oneshot":
        w, h = min(w, 128), min(h, 128)
    while most and w * h > most:
        w, h = (w + 1) // 2, (h + 1) // 2
    if most:
        spp = max(1, min(spp, most // (w * h)))
    c = dict(width=w, height=h, spp=spp, nx=nx, ny=ny, nz=nz)
    if what == "image":
        slices = rng.choice([1, 1, 2, 3])
        return _case(None, kind="draw" if slices == 1 else "progressive", slices=slices,
                     **dict(c, spp=max(1, spp // slices) * slices), nquads=rng.randint(1, 16),
                     preset=1, repeat=rng.random() < 0.3,
                     spectrum=rng.choice(["sw", "sw", "sw_band"]))
    if what == "lw_flux":
        return _case(None, preset=2, sensor="rectangle", spectrum="lw", nquads=rng.randint(2, 16), **c)
    if what == "lw_image":
        return _case(None, preset=2, spectrum="lw", nquads=rng.randint(2, 16), **c)
    if what == "cie":
        return _case(None, preset=1, spectrum="cie", **c)
    if what == "terrain":
        return _case(None, preset=4, sensor=rng.choice(["rectangle", "camera"]),
                     hf_res=_log_int(rng, 33, 512), repeat=rng.random() < 0.3, **c)
    if what == "batch":
        lo, hi = 8 * rng.randint(4, 10), 8 * rng.randint(16, 32)
        return _case(None, kind="batch", scenes=rng.randint(2, 10), width=lo, height=hi,
                     spp=16 * rng.randint(1, 3), nx=32, ny=2 * rng.randint(32, 128))
    if what == "fp64":
        lw = rng.random() < 0.5
        return _case(None, solver="fp64", preset=2 if lw else 1, spectrum="lw" if lw else "sw",
                     nquads=rng.randint(1, 16), sensor=rng.choice(["camera", "rectangle"]),
                     repeat=rng.random() < 0.25, **c)
    return _case(None, kind="oneshot", preset=4, sensor="rectangle", hf_res=_log_int(rng, 33, 512),
                 repeat=rng.random() < 0.5, **c)


def _synth(case, seed):
    """The case's scene: 100 m cells, the cloud base at 1 km, a configuration's
    bands and gas."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    kw = dict(cloud_def=(nx, ny, nz), cloud_upper=(100.0 * nx, 100.0 * ny, 1000.0 + nz * _dz(case)),
              nquads=case["nquads"])
    if case["spectrum"] in ("cie", "sw_band"):
        kw.update(nbands=4, wlen_lo=380.0, wlen_hi=780.0)
    if case["hf_res"]:
        kw["hf_res"] = case["hf_res"]
    s = A.Synth(case["preset"], seed=seed, **kw)
    if case["repeat"]:
        s.scene.repeat_clouds = 1
        s.scene.repeat_ground = 1
    return s


def _dz(case):
    """Cell height: that of the configurations (3.2 km of cloud layer in 32 or
    64 cells, 50 m for the terrain's)"""
    return 3200.0 / case["nz"] if case["preset"] != 4 else 50.0


def _desc(case, seed):
    """The map over the whole grid: a camera south of it looking down across
    it, or a flux rectangle at 2 km."""
    ext = (100.0 * case["nx"], 100.0 * case["ny"], 1000.0 + case["nz"] * _dz(case))
    kw = dict(width=case["width"], height=case["height"], spp=case["spp"] // case["slices"],
              solver=SOLVERS[case["solver"]], seed=seed)
    if case["sensor"] == "camera":
        tilt = math.radians(60.0)
        pos = (ext[0] / 2, -2000.0, ext[2] + 800.0)
        d = A.map_preset(1, pos=pos, **kw,
                         tgt=(pos[0], pos[1] + math.cos(tilt), pos[2] - math.sin(tilt)))
    else:
        d = A.map_preset(4, pos=(ext[0] / 2, ext[1] / 2, 2000.0), rect_size=ext[:2],
                         tgt=(ext[0] / 2, ext[1] / 2, 2001.0), **kw)
    if case["spectrum"] == "lw":
        d.spectral_type = F.SPECTRAL_LW
        d.wlen_range[0], d.wlen_range[1] = 4000.0, 20000.0
        d.ref_temperature = 290.0
    elif case["spectrum"] in ("cie", "sw_band"):
        d.spectral_type = F.SPECTRAL_SW_CIE_XYZ if case["spectrum"] == "cie" else F.SPECTRAL_SW
        d.wlen_range[0], d.wlen_range[1] = 380.0, 780.0
    return d


def _batch_sizes(case):
    """(nx, ny, nz, image side, spp, k-points) of each scene of a batch"""
    rng = np.random.default_rng(case["scenes"] * 1000 + case["ny"])
    out = []
    for _ in range(case["scenes"]):
        nx, ny = (2 * int(rng.integers(case["nx"] // 2, case["ny"] // 2 + 1)) for _ in range(2))
        side = 8 * int(rng.integers(case["width"] // 8, case["height"] // 8 + 1))
        spp = 4 * int(rng.integers(1, case["spp"] // 4 + 1))
        out.append((nx, ny, 2 * int(rng.integers(16, 49)), side, spp, int(rng.integers(1, 17))))
    return out


class _Batch:
    """Scenes, contexts, accumulators and the plan of a batch"""

    def __init__(self, case, seed):
        self.synths, self.descs, self.bufs, items = [], [], [], []
        for i, (nx, ny, nz, side, spp, nq) in enumerate(_batch_sizes(case)):
            c = dict(case, nx=nx, ny=ny, nz=nz, width=side, height=side, spp=spp, nquads=nq)
            self.synths.append(_synth(c, seed * 100 + i))
            self.descs.append(_desc(c, seed * 100 + i))
            self.bufs.append(H.DeviceBuffer(side * side * A.ACCUM_DTYPE.itemsize))
        self.ctxs = [A.Context(s.scene_ptr) for s in self.synths]
        items = [(c, d, b.address) for c, d, b in zip(self.ctxs, self.descs, self.bufs)]
        self.stream = H.Stream()
        self.plan = A.BatchPlan(items)


def prepare(case, seed):
    if case["kind"] == "batch":
        return {"case": case, "batch": _Batch(case, seed)}
    st = {"case": case, "synth": _synth(case, seed), "desc": _desc(case, seed)}
    if case["kind"] != "oneshot":
        st["ctx"] = A.Context(st["synth"].scene_ptr)
    if case["kind"] == "progressive":
        st["accum"] = H.DeviceBuffer(case["width"] * case["height"] * A.ACCUM_DTYPE.itemsize)
        st["stream"] = H.Stream()
    return st


def _results(pixels, desc):
    """The estimates of a map and its counts"""
    names = [k for k in pixels.dtype.names if k not in ("time_sum", "time_sum2", "time_nfail")]
    if desc.sensor == F.SENSOR_CAMERA and desc.spectral_type == F.SPECTRAL_SW:
        names = [k for k in names if not k.startswith("temperature")]
    return {k: pixels[k] for k in names}


def _fetch(buf, desc):
    acc = buf.download(np.empty(desc.width * desc.height, A.ACCUM_DTYPE))
    return _results(A.finalize(desc, acc), desc)


def run(state):
    case = state["case"]
    if case["kind"] == "draw":
        return _results(state["ctx"].draw_map(state["desc"]), state["desc"])
    if case["kind"] == "oneshot":
        with A.Context(state["synth"].scene_ptr) as ctx:
            return _results(ctx.draw_map(state["desc"]), state["desc"])
    if case["kind"] == "progressive":
        d, s = state["desc"], state["stream"]
        state["accum"].zero()
        for k in range(case["slices"]):
            d.spp_offset = k * d.spp
            state["ctx"].render_accum(d, state["accum"].address, s.h.value)
        s.synchronize()
        return _fetch(state["accum"], d)
    b = state["batch"]
    for buf in b.bufs:
        buf.zero()
    b.plan.rewind()
    b.plan.step(b.stream.h.value)
    b.stream.synchronize()
    return [_fetch(buf, d) for buf, d in zip(b.bufs, b.descs)]


def _one_work(case):
    pixels = case["width"] * case["height"]
    channels = 3 if case["spectrum"] == "cie" else 1
    spp = case["spp"] // case["slices"] * case["slices"]
    ops = OPS["terrain" if case["hf_res"] else "lw" if case["spectrum"] == "lw" else "sw"]
    cells = case["nx"] * case["ny"] * case["nz"]
    tris = 2 * max(case["hf_res"] - 1, 0) ** 2
    # the cloud grid, one 8-byte octree record per 2^3 cells, the triangles
    # and their boxes, the pixels
    nbytes = 4 * cells + cells + (36 + 16) * tris + 64 * channels * pixels
    return {"bytes": nbytes, "flops": pixels * spp * channels * ops}


def work(case):
    if case["kind"] != "batch":
        return _one_work(case)
    total = {"bytes": 0, "flops": 0.0}
    for nx, ny, nz, side, spp, nq in _batch_sizes(case):
        w = _one_work(dict(case, nx=nx, ny=ny, nz=nz, width=side, height=side, spp=spp, nquads=nq))
        total = {k: total[k] + w[k] for k in total}
    return total


def exact(case, seed):
    """None: a pixel is the mean of random walks, each some hundred dependent
    collisions long. Their value in 64 bits is another run of every walk, with
    its random stream, one collision at a time, which plain numpy does not do
    in 20 s."""
    return None
