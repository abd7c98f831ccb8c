"""Nodal states between CATHY's order and the device rows, bit for bit: meshes
on either side of the 50,000 nodes up to which the host permutes what it reads
(the largest also with rows in tiles and in the natural order)."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_tiles import _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,layers,order", [
    (1, 1, 1, 1), (9, 8, 5, 0), (49, 49, 19, 1), (49, 50, 19, 1), (49, 50, 20, 2), (60, 50, 20, 3), (60, 50, 20, 0)])
def test_states_round_trip(rows, cols, layers, order):
    from pycathy_wrapper_amd import gpu as G
    pr = _problem(rows, cols, layers, 1)
    f = G.FlowGPU(pr, order)
    try:
        f.init(pr.psi0)
        assert np.array_equal(f.psi(), pr.psi0)   # dry surface: INIT leaves every head
        psi = np.random.default_rng(rows).standard_normal(pr.mesh.n)
        f.set_pnew(psi)
        assert np.array_equal(f.psi(), psi)
    finally:
        f.close()
