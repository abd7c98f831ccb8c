"""Which form of the solver a mesh gets (CPU, the HIP calls on host memory:
hip_host_stub.c).  Meshes that need more tiles than there are CUs run on them only with
one row per thread.  Every case of test_gpu_tiles runs on tiles with the rows per
thread it is a test of, and chain-major rows run on none."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

from test_alloc_failure import ROOT, stub  # noqa: F401

PROG = r"""
import test_gpu_tiles as T
from pycathy_wrapper_amd import gpu as G
cases = [m for m in T.test_tiles_match_oracle_and_colour_launches.pytestmark if m.name == "parametrize"][0].args[1]
small = {c[:3] for c in cases if c[0] * c[1] * c[2] < 100000} | {(12, 12, 28)}
for sz in sorted(small):
    f = G.FlowGPU(T._problem(*sz, 1), G.ORDER_COLUMN3)
    assert T._on_tiles(f, *sz), (sz, f.tiles())
    assert f.tiles()["threads"] <= 1024 and f.tiles()["threads"] % 64 == 0
    c = G.FlowGPU(T._problem(*sz, 1), G.ORDER_COLUMN3C)
    assert c.tiles() == dict(tiles=0, rows_per_thread=0, threads=0, last=False), sz
assert len(small) > 8 and any(sz in T.TWO_ROWS for sz in small)
"""


def test_the_tile_cases_take_the_form_they_test(stub):  # noqa: F811
    r = subprocess.run([sys.executable, "-c", PROG], cwd=ROOT, capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, LD_PRELOAD=stub, PYTHONPATH=ROOT + ":" + os.path.join(ROOT, "tests")))
    assert r.returncode == 0, r.stderr


# one tile per CU at most with two rows per thread; more with two: none; more with one
@pytest.mark.parametrize("rows,cols,layers,tiles,rpt", [(126, 126, 14, (1, 256), 2), (130, 130, 13, (0, 0), 0),
                                                        (135, 135, 12, (257, 400), 1)])
def test_more_tiles_than_cus_need_one_row_per_thread(stub, rows, cols, layers, tiles, rpt):  # noqa: F811
    prog = f"import test_gpu_tiles as T\nfrom pycathy_wrapper_amd import gpu as G\n" \
           f"t = G.FlowGPU(T._problem({rows}, {cols}, {layers}, 1), 1).tiles()\n" \
           f"assert {tiles[0]} <= t['tiles'] <= {tiles[1]} and t['rows_per_thread'] == {rpt}, t\n"
    r = subprocess.run([sys.executable, "-c", prog], cwd=ROOT, capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, LD_PRELOAD=stub, PYTHONPATH=ROOT + ":" + os.path.join(ROOT, "tests")))
    assert r.returncode == 0, r.stderr
