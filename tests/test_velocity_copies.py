"""How the nodal velocities reach the caller (CPU, the HIP calls on host memory:
hip_host_stub.c).  Up to 50,000 nodes they pass through one array of the
library's, which is faster than copies into three arrays that the caller has
just made; beyond, the copies go to the caller directly."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

from test_alloc_failure import ROOT, stub  # noqa: F401

PROG = r"""
import ctypes as C, sys
import numpy as np
from pycathy_wrapper_amd import gpu as G
from test_gpu_tiles import _problem
lib = C.CDLL(None)
lib.hip_stub_copies.argtypes = [C.c_void_p]
f = G.FlowGPU(_problem(*map(int, sys.argv[1:4]), 1))
out = f.velocity()
n = [lib.hip_stub_copies(out[k].ctypes.data) for k in ("unod", "vnod", "wnod")]
assert len(set(n)) == 1, n
print(n[0])
"""


@pytest.mark.parametrize("rows,cols,layers,direct", [(4, 5, 3, 0), (49, 49, 19, 0), (49, 50, 20, 1)])
def test_nodal_velocities_of_small_meshes_take_the_warm_array(stub, rows, cols, layers, direct):  # noqa: F811
    r = subprocess.run([sys.executable, "-c", PROG, str(rows), str(cols), str(layers)], cwd=ROOT, capture_output=True,
                       text=True, timeout=120,
                       env=dict(os.environ, LD_PRELOAD=stub, PYTHONPATH=ROOT + ":" + os.path.join(ROOT, "tests")))
    assert r.returncode == 0, r.stderr
    assert int(r.stdout.split()[-1]) == direct
