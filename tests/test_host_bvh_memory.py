"""A ground mesh whose BVH finds no memory is an error of the call, on whichever
thread it happens, and not the end of the process."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CODE = """
import resource
import sys
import numpy as np
from htrdr_kmin_amd import _ffi as F
from htrdr_kmin_amd import atmosphere as A

def scene(hf_res):
    return A.Synth(4, seed=1, hf_res=hf_res, cloud_def=(32, 32, 32), cloud_upper=(3200.0, 3200.0, 4200.0))

rays = np.array([[10.0, 10.0, 5000.0, 0.0, 0.0, -1.0, 0.0, 1e9]])
small, big = scene(120), scene(700)
A.mesh_trace(small.scene_ptr, rays)  # the threads run
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
got = []
for mb in MBS:
    resource.setrlimit(resource.RLIMIT_AS, (used + (mb << 20), resource.RLIM_INFINITY))
    try:
        A.mesh_trace(big.scene_ptr, rays)
        got.append("ok")
    except F.HtgxError as e:
        assert e.code == F.MEM_ERR
        got.append("no memory")
print(got)
assert got[0] == "no memory" and got[-1] == "ok"
"""


@pytest.mark.parametrize("threads", [1, 7])
def test_no_memory_is_an_error(threads):
    env = dict(os.environ, OMP_NUM_THREADS=str(threads))
    code = CODE.replace("MBS", repr(list(range(8, 200, 4)) + [1000]))
    r = subprocess.run([sys.executable, "-c", code], env=env, cwd=ROOT, capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
