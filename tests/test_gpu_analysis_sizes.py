"""The analysis kernels at the edges of their member widths (8, 16, 32, 64: one
below, at and above), of the localised kernel's LDS fill (2,048 values: 256 to 32
observations) and of its groups of four observations, in every localisation, against
numpy in extended precision; then the members' continuation from the analysis,
which one launch takes for all, against a run started from that state.

Bound of the analysis: a sum of m products per member, each of a dot over the members,
so (m + members) roundings of the largest partial sum; 1e-12 of the largest
state is four orders above that at m = 300.  Sw and kr of a continued state come
from the functions that a started run takes them from: the same bits.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from test_gpu_tiles import _problem

pytestmark = pytest.mark.gpu


def _members(n, rows=6, cols=7, layers=4):
    from pycathy_wrapper_amd import gpu as G
    pr = _problem(rows, cols, layers, 1)
    rng = np.random.default_rng(n)
    flows = [G.FlowGPU(pr, G.ORDER_COLUMN3) for _ in range(n)]
    X = []
    for f in flows:
        f.init(pr.psi0)
        X.append(pr.psi0 + 0.1 * rng.standard_normal(pr.mesh.n))
        f.set_pnew(X[-1])
    return pr, flows, np.stack(X, axis=1).astype(np.longdouble), rng


def _zones(flows, S, invD, zr, zo, alpha):
    from pycathy_wrapper_amd import gpu as G
    h = np.array([f.h.value for f in flows], dtype=np.int64)
    zr, zo = zr.astype(np.int32), zo.astype(np.int32)
    G._check(G.lib().cathy_gpu_enkf_update_zones(G._i(len(flows)), G._p(h), G._i(len(S)), G._p(S), G._p(invD),
                                                 G._p(zr), G._p(zo), C.byref(C.c_double(alpha))), "zones")


def _inflate(xa, alpha):
    mean = xa.mean(axis=1, keepdims=True)
    return mean + alpha * (xa - mean)


@pytest.mark.parametrize("n,m,mode,alpha", [
    (2, 1, "dense", 1.0), (7, 3, "xy", 1.1), (8, 257, "dense", 1.0), (9, 4, "zones", 1.0), (16, 129, "xy", 1.0),
    (17, 5, "dense", 1.2), (32, 64, "zones", 1.1), (33, 33, "xy", 1.0), (64, 70, "dense", 1.0), (24, 300, "xy", 1.0)])
def test_localised_analysis(n, m, mode, alpha):
    from pycathy_wrapper_amd import enkf as EK
    pr, flows, X, rng = _members(n)
    try:
        S, invD = rng.standard_normal((m, n)), rng.standard_normal((m, n))
        obs = rng.integers(0, pr.mesh.n, m)
        xy = np.stack([pr.mesh.x, pr.mesh.y], axis=1)
        if mode == "dense":
            L = rng.uniform(0.0, 1.0, (pr.mesh.n, m))
            EK.enkf_update_localized(flows, S, invD, L=L, inflation=alpha)
        elif mode == "xy":
            L = EK.gaspari_cohn(np.linalg.norm(xy[:, None] - xy[obs][None], axis=2), 4.0)
            EK.enkf_update_localized(flows, S, invD, obs_xy=xy[obs], radius=4.0, inflation=alpha)
        else:
            zr, zo = np.arange(pr.mesh.n) % 5, rng.integers(0, 4, m)   # zone 4 holds no observation
            L = (zr[:, None] == zo[None]).astype(float)
            _zones(flows, S, invD, zr, zo, alpha)
        Xp = X - X.mean(axis=1, keepdims=True)
        xa = _inflate(X + ((Xp @ S.T.astype(np.longdouble)) / (n - 1) * L) @ invD.astype(np.longdouble), alpha)
        if mode == "zones":
            still = ~L.any(axis=1)
            xa[still] = X[still]
        got = np.stack([f.psi() for f in flows], axis=1)
        assert np.max(np.abs(got - xa)) <= 1e-12 * np.max(np.abs(xa))
        for j in (0, n - 1):
            sw, kr = flows[j].sw(), flows[j].ckrw()
            flows[j].init(got[:, j])
            assert np.array_equal(flows[j].psi(), got[:, j])
            assert np.array_equal(flows[j].sw(), sw) and np.array_equal(flows[j].ckrw(), kr)
    finally:
        for f in flows:
            f.close()


@pytest.mark.parametrize("n,alpha", [(2, 1.0), (8, 1.1), (9, 1.0), (32, 1.0), (33, 1.1), (64, 1.0)])
def test_global_analysis(n, alpha):
    from pycathy_wrapper_amd import enkf as EK
    pr, flows, X, rng = _members(n)
    try:
        W = rng.standard_normal((n, n)) / n
        EK.enkf_update(flows, W, alpha)
        xa = _inflate(X + (X - X.mean(axis=1, keepdims=True)) @ W.astype(np.longdouble), alpha)
        got = np.stack([f.psi() for f in flows], axis=1)
        assert np.max(np.abs(got - xa)) <= 1e-12 * np.max(np.abs(xa))
    finally:
        for f in flows:
            f.close()
