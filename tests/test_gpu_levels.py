"""The natural order's level kernels (IC(0) factor and sweeps) at the sizes
where their launch rule changes, against the C oracle's SYMSLV.

The factor runs in one work-group up to levels of 512 rows, the sweeps in
one work-group (1024 threads) while the reach of a row plus the longest level
fit the 8,192-row LDS ring, both only for rows of at most 8 entries on
either side of the diagonal.  The systems are diagonally dominant, so the
same NITER follows from the same recurrences; the solution's bound is
that of test_gpu_parity (1e-12, the sums differ in order only).
"""
from __future__ import annotations

import numpy as np
import pytest

from pycathy_wrapper_amd import mesh as ME
import systems as SY

pytestmark = pytest.mark.gpu


def _extruded(rows, cols, layers):
    m = ME.build_mesh(100.0 - 0.1 * np.arange(cols)[None, :] + np.zeros((rows, 1)), 2.0, 2.0, layers,
                      np.full(layers, 1.0 / layers), 5.0)
    topol, ja = ME.sym_pattern(m.tetra, m.n)
    return topol, ja


def _random_pattern(n, per_row, seed):
    """Upper CSR with random couplings: rows of up to a dozen lower entries."""
    rng = np.random.default_rng(seed)
    r = np.repeat(np.arange(n), per_row)
    c = r + rng.integers(-60, 61, r.size)
    ok = (c >= 0) & (c < n)
    lo, hi = np.minimum(r, c)[ok], np.maximum(r, c)[ok]
    key = np.unique(np.concatenate([lo[lo < hi] * n + hi[lo < hi], np.arange(n) * (n + 1)]))
    return np.searchsorted(key, np.arange(n + 1) * n).astype(np.int32), (key % n).astype(np.int32)


def _values(topol, ja, seed):
    """Random negative couplings, diagonal 1.05 times the row's sum."""
    rng = np.random.default_rng(seed)
    n = len(topol) - 1
    row = np.repeat(np.arange(n), np.diff(topol))
    v = -np.exp(rng.normal(0.0, 1.0, len(ja)))
    v[row == ja] = 0.0
    s = -(np.bincount(row, v, n) + np.bincount(ja, v, n))
    v[topol[:-1]] = 1.05 * s + 0.1
    return v, rng.standard_normal(n)


def _check(gpu, oracle, topol, ja, nod0, seed):
    v, b = _values(topol, ja, seed)
    nd1 = None
    if nod0 is not None:
        v, b = v.copy(), b.copy()
        v[topol[nod0]] *= 1e-9 * 1.7e100
        b[nod0] = 0.0
        nd1 = (nod0 + 1).astype(np.int32)
    x, it, err, res, _ = SY.oracle_symslv(oracle, topol, ja, v, b, nod0)
    xg, itg, errg, resg, rc = gpu.symslv(topol + 1, ja + 1, v, b, nd1)
    assert rc == 0 and itg == it, (itg, it)
    assert np.max(np.abs(xg - x)) <= 1e-12 * np.max(np.abs(x))
    assert errg == pytest.approx(err, rel=1e-6)


@pytest.fixture(scope="module")
def gpu():
    from pycathy_wrapper_amd import gpu as G
    yield G
    G.symslv_release()


# levels of 1 row (a single column), a few, 77, 845 (factor level by level), 1,331 rows (more
# than one row per thread), and past the ring (level by level throughout)
@pytest.mark.parametrize("rows,cols,layers", [(1, 1, 1), (3, 2, 4), (10, 70, 6), (64, 48, 20), (70, 72, 24),
                                              (125, 125, 26)])
def test_level_kernels_match_oracle(gpu, oracle, rows, cols, layers):
    topol, ja = _extruded(rows, cols, layers)
    n = len(topol) - 1
    _check(gpu, oracle, topol, ja, None, 3)
    _check(gpu, oracle, topol, ja, np.arange(0, n, 7, dtype=np.int64), 4)


@pytest.mark.parametrize("n,per_row", [(400, 2), (3000, 6)])
def test_irregular_rows_match_oracle(gpu, oracle, n, per_row):
    """Rows within the tables' eight lower entries (per_row 2) and beyond."""
    topol, ja = _random_pattern(n, per_row, 5)
    _check(gpu, oracle, topol, ja, None, 6)
    _check(gpu, oracle, topol, ja, np.arange(0, n, 9, dtype=np.int64), 7)
