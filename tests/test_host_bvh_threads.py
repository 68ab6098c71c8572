"""The ground BVH does not depend on the threads it is built with: distances,
triangles and the number of nodes visited by rays through terrains below and
above the size from which a node's own passes run on all threads."""
import hashlib
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def digest(hf_res):
    from htrdr_kmin_amd import atmosphere as A
    rng = np.random.default_rng(hf_res)
    s = A.Synth(4, seed=hf_res, hf_res=hf_res, cloud_def=(32, 32, 32), cloud_upper=(3200.0, 3200.0, 4200.0))
    n = 2000
    o = rng.uniform([0, 0, -100], [3200, 3200, 3000], (n, 3))
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    rays = np.concatenate([o, d, np.zeros((n, 1)), np.full((n, 1), 1e9)], 1)
    h = hashlib.sha256()
    for x in A.mesh_trace(s.scene_ptr, rays):
        h.update(np.ascontiguousarray(x).tobytes())
    return h.hexdigest()


@pytest.mark.parametrize("hf_res", [2, 33, 91, 92, 200, 400])
def test_tree_does_not_depend_on_threads(hf_res):
    got = set()
    for threads in (1, 2, 7):
        env = dict(os.environ, OMP_NUM_THREADS=str(threads))
        code = f"import sys; sys.path[:0]=[{ROOT!r}, {ROOT + '/tests'!r}]; " \
               f"import test_host_bvh_threads as T; print(T.digest({hf_res}))"
        got.add(subprocess.run([sys.executable, "-c", code], env=env, check=True, capture_output=True,
                               text=True).stdout.strip().splitlines()[-1])
    assert len(got) == 1
