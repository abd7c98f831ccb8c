"""A device allocation that fails while a buffer grows (CPU, the HIP calls on
host memory: hip_host_stub.c): the call reports it, and the next call of a
smaller size works on buffers that exist.  Each allocation of the larger call
fails in turn; the later call must leave as many buffers held as the first one did.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PROG = r"""
import ctypes as C, gc, sys
import numpy as np
from pycathy_wrapper_amd import configs as CF, enkf as EN, gpu as G, guess as GN, mesh as ME, routing as RO
stub = C.CDLL(None)

def case_route():
    net = RO.synthetic_network(9, 7)
    state = lambda m: {k: np.zeros((m, net.ngrid)) for k in RO.STATE_IN + RO.STATE_INOUT + RO.STATE_OUT}
    r = RO.RouteGPU(net)
    return lambda big: r.step(1.0, state(5 if big else 2))

def case_gradient(levels):
    lp = GN.padded(levels)
    net = GN.GuessNet(levels, seed=0)
    def call(big):
        m = 300 if big else 20
        net.gradient(np.zeros((m, lp, GN.NFEAT), np.uint16), np.zeros((m, lp), np.float32))
    return call

def case_train():
    net = GN.GuessNet(16, seed=0)
    load = lambda m: net.load(np.zeros((m, 16, GN.NFEAT), np.uint16), np.zeros((m, 16), np.float32))
    state = dict(failed=False)
    def call(big):
        if big:  # a set whose load fails is gone: no steps on it
            state["failed"] = True
            load(300)
            state["failed"] = False
        elif state["failed"]:
            try:
                net.train(2, 16)
                raise AssertionError("steps without a training set")
            except G.CathyGpuError as e:
                assert "no training set" in str(e), e
        if not big:
            load(20)
        net.train(2, 16)
    return call

def case_analysis():
    m = ME.build_mesh(100.0 + np.zeros((3, 4)), 1.0, 1.0, 3, np.full(3, 1.0 / 3.0), 1.0)
    one = lambda v: np.full((3, 1), v)
    soil = dict(nzone=1, permx=one(1e-5), permy=one(1e-5), permz=one(1e-5), elstor=one(1e-4), poros=one(0.4),
                vgn=one(1.5), vgrmc=one(0.05), vgpsat=one(1.0))
    pr = CF.Problem("alloc", m, soil, CF.icvdwt(m, 0.5), np.array([0.0]), np.array([0.0]), CF.hillslope_small_params(), 0)
    flows = [G.FlowGPU(pr) for _ in range(9)]
    def call(big):
        k = 9 if big else 2
        h = np.array([f.h.value for f in flows[:k]], dtype=np.int64)
        G._check(G.lib().cathy_gpu_enkf_update(G._i(k), G._p(h), G._p(np.zeros((k, k))),
                                               C.byref(C.c_double(1.0))), "enkf_update")
    return call

def case_velocity():
    m = ME.build_mesh(100.0 + np.zeros((3, 4)), 1.0, 1.0, 3, np.full(3, 1.0 / 3.0), 1.0)
    one = lambda v: np.full((3, 1), v)
    soil = dict(nzone=1, permx=one(1e-5), permy=one(1e-5), permz=one(1e-5), elstor=one(1e-4), poros=one(0.4),
                vgn=one(1.5), vgrmc=one(0.05), vgpsat=one(1.0))
    pr = CF.Problem("alloc", m, soil, CF.icvdwt(m, 0.5), np.array([0.0]), np.array([0.0]), CF.hillslope_small_params(), 0)
    f = G.FlowGPU(pr)
    return lambda big: f.velocity()

make = dict(route=case_route, gradient=lambda: case_gradient(16), gradient_deep=lambda: case_gradient(70),
            train=case_train, analysis=case_analysis, velocity=case_velocity)[sys.argv[1]]
def held(make):
    # buffers the objects of a case hold after a call of the small size
    base = stub.hip_stub_live()
    c = make()
    c(False)
    n = stub.hip_stub_live() - base
    del c
    gc.collect()
    assert stub.hip_stub_live() == base
    return n

want, k = held(make), 0
while True:  # allocation k of the larger call fails, until the call has no more
    base = stub.hip_stub_live()
    c = make()
    if sys.argv[1] != "velocity":  # (its buffers are allocated by the first call)
        c(False)
    stub.hip_stub_fail(k)
    try:
        c(True)
        break
    except G.CathyGpuError as e:
        assert "(-3)" in str(e), e
    stub.hip_stub_fail(-1)
    c(False)
    assert stub.hip_stub_live() - base >= want, f"buffers missing after allocation {k} failed"
    del c
    gc.collect()
    k += 1
assert k > 0
print("allocations of the larger call:", k)
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    if shutil.which("gcc") is None or not os.path.exists(os.path.join(ROOT, "pycathy_wrapper_amd", "libcathy_gpu.so")):
        pytest.skip("needs gcc and the built library")
    so = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "hip_host_stub.c")], check=True)
    return so


@pytest.mark.parametrize("case", ["route", "gradient", "gradient_deep", "train", "analysis", "velocity"])
def test_a_failed_allocation_leaves_nothing_half_sized(stub, case):
    r = subprocess.run([sys.executable, "-c", PROG, case], cwd=ROOT, capture_output=True, text=True, timeout=120,
                       env=dict(os.environ, LD_PRELOAD=stub, PYTHONPATH=ROOT))
    assert r.returncode == 0, r.stdout + r.stderr
