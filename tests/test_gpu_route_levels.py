"""Routing networks that take each form of the level loop, against the C oracle:
four cells, a strip (levels of one cell), a wide grid whose levels exceed one
pass of cells (256), grids with part of the branches cut, whose cells join far below
their level (feeders many levels back), and one of these with more outflows
waiting for their readers than the 7,168 LDS slots.  Tolerance of
test_gpu_route."""
from __future__ import annotations

import numpy as np
import pytest

from pycathy_wrapper_amd import routing as RT
from test_gpu_route import _compare
from test_oracle_route import advance, initial_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,cut,members", [(2, 2, 0.0, 1), (1, 60, 0.0, 2), (300, 300, 0.0, 1), (60, 45, 0.3, 3),
                                                   (300, 299, 0.6, 1)])
def test_level_forms(rows, cols, cut, members):
    import pyoracle as P
    net = RT.synthetic_network(rows, cols, dx=10.0, seed=rows)
    if cut:  # headwaters at any level: the cell's water stays on it
        lost = np.random.default_rng(cols).uniform(size=net.w1.shape) < cut
        lost.ravel()[0] = False
        net.w1[lost] = 0.0
        net.w2[lost] = 0.0
    g = RT.RouteGPU(net)
    orc = P.Oracle()
    sd = initial_state(net, members)
    so = [{k: (v[m] if members > 1 else v).copy() for k, v in sd.items()} for m in range(members)]
    try:
        for sub in range(2):
            cu_d, ak_d = g.step(30.0, sd)
            res = [orc.route(net, 30.0, st) for st in so]
            _compare(net, sd, so, cu_d, ak_d, [r[0] for r in res], [r[1] for r in res], sub)
            advance(sd)
            for st in so:
                advance(st)
    finally:
        g.close()
