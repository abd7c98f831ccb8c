"""The solver over surface tiles (column ordering, rows plane by plane) at the
sizes where its tiles change, against the C oracle and against the same
ordering with chain-major rows, which takes the five colour launches.

Surfaces of fewer columns than a tile, of exactly one and of one more, long
strips, two planes (no inner plane), columns so deep that the tiles shrink
to fit a work-group (41 and 64 planes), both rows-per-thread forms, both factor
precisions, Picard (PCG) and Newton (BiCGSTAB: separate sweeps).  Both
orderings eliminate the same colours, so the factor has the same entries and the
PCG counts agree but for one iteration per solve whose error lands on the
tolerance's other side.  psi's bound is that of test_gpu_parity.  (Newton on
90x90x22 is no test of this: its first BiCGSTAB solve is marginal, 1,132
iterations with chain-major rows where the oracle, the natural and both other column
orderings step back.)

Each case asserts that it runs on tiles, with the rows per thread it is there for,
and that chain-major rows do not.  The preconditioner itself is compared on one
flow: z of the tiles against z of the colour launches with the same factor, bit for bit,
since a run that shares the GPU with many others takes the launches to the same bits.
Lockstep members on tiles equal their solo runs bit for bit, in both precisions.
"""
from __future__ import annotations

import numpy as np
import pytest

from pycathy_wrapper_amd import configs as CF
from pycathy_wrapper_amd import mesh as ME

pytestmark = pytest.mark.gpu

PSI_TOL = 1e-6


@pytest.fixture(scope="module")
def gpu():
    from pycathy_wrapper_amd import gpu as G
    G.device_info()
    return G


def _problem(rows, cols, layers, iopt):
    rng = np.random.default_rng([rows, cols, layers])
    dem = 100.0 - 0.05 * np.arange(cols)[None, :] + 0.05 * rng.uniform(-1.0, 1.0, (rows, cols))
    nz = rows * cols
    zone = np.arange(1, nz + 1, dtype=np.int32).reshape(rows, cols)
    m = ME.build_mesh(dem, 2.0, 2.0, layers, np.full(layers, 1.0 / layers), 5.0, zone=zone)
    f = lambda v: np.full((layers, nz), v)
    ks = np.exp(np.log(1e-5) + rng.standard_normal((layers, nz)))
    soil = dict(nzone=nz, permx=ks, permy=ks.copy(), permz=ks.copy(), elstor=f(1e-4), poros=f(0.45),
                vgn=f(1.46), vgrmc=f(0.05), vgpsat=f(1.0))
    return CF.Problem("tiles", m, soil, CF.icvdwt(m, 1.0), np.array([0.0]), np.array([5e-7]),
                      CF.hillslope_small_params(iopt=iopt), 0)


TWO_ROWS = {(12, 12, 28), (12, 12, 40), (9, 9, 63), (90, 90, 22)}   # meshes whose phases take two rows per thread


def _on_tiles(f, rows, cols, layers):
    """The flow runs on tiles, as many rows per thread as the mesh is a test of."""
    t = f.tiles()
    return t["tiles"] >= 1 and t["rows_per_thread"] == (2 if (rows, cols, layers) in TWO_ROWS else 1)


@pytest.mark.parametrize("rows,cols,layers,iopt,fp64", [
    (1, 1, 1, 1, False), (1, 30, 2, 1, False), (4, 4, 3, 1, False), (1, 12, 5, 1, True), (5, 4, 3, 2, False),
    (3, 40, 1, 2, False), (9, 31, 5, 1, True), (24, 25, 15, 1, False), (12, 12, 40, 1, False), (12, 12, 40, 2, True),
    (9, 9, 63, 1, False), (85, 86, 2, 1, False), (90, 90, 22, 1, True), (40, 41, 15, 2, False)])
def test_tiles_match_oracle_and_colour_launches(gpu, oracle, rows, cols, layers, iopt, fp64):
    import pyoracle as P
    pr = _problem(rows, cols, layers, iopt)
    m = pr.mesh
    run = oracle.run_create(dict(tetra=m.tetra, x=m.x, y=m.y, z=m.z, arenod=m.arenod, nnod=m.nnod, nstr=m.nstr,
                                 ntri=m.ntri), pr.soil, pr.psi0, pr.atm_times, pr.atm_vals, pr.hspatm,
                            P.OrcParams(**pr.params.as_dict()))
    flows = [gpu.FlowGPU(pr, o) for o in (gpu.ORDER_COLUMN3, gpu.ORDER_COLUMN3C)]
    try:
        for f in flows:
            f.factor_fp64(fp64)
        assert _on_tiles(flows[0], rows, cols, layers) and flows[1].tiles()["tiles"] == 0
        for _ in range(2 if m.n < 50000 else 1):
            _, so = run.step()
            st = [f.advance()[1] for f in flows]
            psi = run.psi()
            for f, s in zip(flows, st):
                assert (s["DELTAT"], s["ITER"], s["BACK"]) == (so["DELTAT"], so["ITER"], so["BACK"])
                assert np.max(np.abs(f.psi() - psi)) <= PSI_TOL * np.max(np.abs(psi))
            assert abs(st[0]["NITERT"] - st[1]["NITERT"]) <= so["ITER"] + 10 * so["BACK"]
    finally:
        run.close()
        for f in flows:
            f.close()


@pytest.mark.parametrize("rows,cols,layers,iopt,fp64", [
    (1, 1, 1, 1, False), (1, 30, 2, 1, True), (5, 4, 3, 2, False), (24, 25, 15, 1, False), (24, 25, 15, 2, True),
    (12, 12, 40, 1, True), (12, 12, 40, 2, False), (9, 9, 63, 1, False), (90, 90, 22, 1, False)])
def test_the_tiles_precondition_as_the_colour_launches(gpu, rows, cols, layers, iopt, fp64):
    pr = _problem(rows, cols, layers, iopt)
    f = gpu.FlowGPU(pr, gpu.ORDER_COLUMN3)
    try:
        f.factor_fp64(fp64)
        assert _on_tiles(f, rows, cols, layers)
        with pytest.raises(gpu.CathyGpuError, match="none has run"):
            f.precond(np.zeros(pr.mesh.n))
        f.advance()
        rng = np.random.default_rng(rows)
        for t in (rng.standard_normal(pr.mesh.n), np.eye(1, pr.mesh.n, pr.mesh.n // 2)[0]):
            z, zl = f.precond(t), f.precond(t, launches=True)
            assert np.any(z != 0.0) and np.all(np.isfinite(z))
            assert np.array_equal(z, zl)
    finally:
        f.close()


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("sizes", [((12, 12, 28), (12, 12, 28)), ((24, 25, 15), (9, 31, 5)),
                                   ((12, 12, 28), (4, 4, 3), (24, 25, 15))])
def test_lockstep_on_tiles_matches_solo_runs(gpu, sizes, fp64):
    """Members with one and two rows per thread in one launch, each its solo run's bits."""
    probs = [_problem(*sz, 1) for sz in sizes]
    for k, pr in enumerate(probs):
        pr.psi0 = pr.psi0 - 0.01 * k
    flows = [gpu.FlowGPU(pr, gpu.ORDER_COLUMN3) for pr in probs]
    for f, sz in zip(flows, sizes):
        f.factor_fp64(fp64)
        assert _on_tiles(f, *sz)
    ens = gpu.EnsembleGPU(flows)
    try:
        rc, taken, stats = ens.advance(2)
        assert np.all(rc == 0) and np.all(taken == 2)
        psi = [f.psi() for f in flows]
    finally:
        ens.close()
        for f in flows:
            f.close()
    for pr, st, ps in zip(probs, stats, psi):
        f = gpu.FlowGPU(pr, gpu.ORDER_COLUMN3)
        try:
            f.factor_fp64(fp64)
            for s in st:
                assert f.advance()[1] == s
            assert np.array_equal(f.psi(), ps)
        finally:
            f.close()


def _solo(gpu, pr, fp64, steps):
    f = gpu.FlowGPU(pr, gpu.ORDER_COLUMN3)
    try:
        f.factor_fp64(fp64)
        st = [f.advance()[1] for _ in range(steps)]
        assert f.tiles()["last"]     # alone, over tiles
        return st, f.psi()
    finally:
        f.close()


@pytest.mark.parametrize("members,fp64,graphs", [(3, False, False), (9, False, False), (9, True, True)])
def test_a_full_gpu_takes_the_launches_to_the_same_bits(gpu, members, fp64, graphs):
    """26,896-node members: three in lockstep run over tiles, nine (242,064
    rows) by the colour launches; every step is the solo run's, bit for bit."""
    probs = [_problem(40, 40, 15, 1) for _ in range(members)]
    for k, pr in enumerate(probs):
        pr.psi0 = pr.psi0 - 0.01 * k
    flows = [gpu.FlowGPU(pr, gpu.ORDER_COLUMN3) for pr in probs]
    for f in flows:
        f.factor_fp64(fp64)
    ens = gpu.EnsembleGPU(flows)
    try:
        ens.graphs(graphs)
        rc, taken, stats = ens.advance(2)
        assert np.all(rc == 0) and np.all(taken == 2)
        assert ens.tile_rounds() == (ens.info()["rounds"] if members == 3 else 0)
        assert all(f.tiles()["tiles"] > 0 and f.tiles()["last"] == (members == 3) for f in flows)
        psi = [f.psi() for f in flows]
    finally:
        ens.close()
        for f in flows:
            f.close()
    for j in (0, members - 1):
        st, ps = _solo(gpu, probs[j], fp64, 2)
        assert st == stats[j] and np.array_equal(ps, psi[j])


@pytest.mark.parametrize("iopt", [1, 2])
def test_runs_on_threads_match_runs_alone(gpu, iopt):
    """Four 63,257-node runs on threads of their own fill the GPU past the
    tiles' line at times; whichever way a solve takes, the bits are the solo run's."""
    import threading
    pr = _problem(60, 60, 16, iopt)
    want, psi = _solo(gpu, pr, False, 2)
    flows = [gpu.FlowGPU(pr, gpu.ORDER_COLUMN3) for _ in range(4)]
    got = [None] * 4
    start = threading.Barrier(4)

    def run(i):
        start.wait()
        got[i] = [flows[i].advance()[1] for _ in range(2)]

    try:
        th = [threading.Thread(target=run, args=(i,)) for i in range(4)]
        for t in th:
            t.start()
        for t in th:
            t.join()
        for i in range(4):
            assert got[i] == want and np.array_equal(flows[i].psi(), psi)
    finally:
        for f in flows:
            f.close()
