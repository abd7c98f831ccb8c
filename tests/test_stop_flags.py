"""The solvers' stop flags in the kernel sources (CPU).

A work-group that returns before its barriers on a flag which another group of
the same launch stores can split: some waves see the old value and wait at the
barrier, the others are gone, and the sums that the rest form in LDS lack their
parts.  No run shows it reliably, so the sources are read: a kernel (or the
device function it is made of) that reads a stop flag does not store the same flag,
unless every launch of it is one work-group whose waves all read the flag
ahead of the barrier that comes before the store.
"""
from __future__ import annotations

import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pycathy_wrapper_amd", "csrc")
FLAGS = {"done": r"\*(?:P\.)?done\b", "stop": r"\b(?:P\.)?sc->stop\b"}
ONE_GROUP = {"pcg_check_body": ("k_pcg_check", "kb_pcg_check"), "k_bicg_check": ("k_bicg_check",)}


def _functions():
    """(name, body) of every device function and kernel of the solver sources."""
    for f in sorted(glob.glob(os.path.join(CSRC, "*.hip"))):
        src = re.sub(r"//[^\n]*", "", open(f).read())
        for m in re.finditer(r"^(?:template[^\n]*\n)?(?:__device__|__global__)[^;{]*?\b(\w+)\(([^{;]*)\)\s*\{", src, re.M):
            depth, i = 1, m.end()
            while depth:
                depth += {"{": 1, "}": -1}.get(src[i], 0)
                i += 1
            yield m.group(1), src[m.end():i]


def _reads_and_stores(body):
    """Flags the body reads (not only as the target of a store), flags it stores."""
    reads, stores = set(), set()
    for name, pat in FLAGS.items():
        store = pat + r"\s*=(?!=)"
        if re.search(store, body):
            stores.add(name)
        if re.search(pat, re.sub(store, "", body)):
            reads.add(name)
    return reads, stores


def test_the_solvers_flags_are_found():
    found = {n: _reads_and_stores(b) for n, b in _functions()}
    for n in ("spmv_beta_body", "tile_body", "pcg_check_body", "pcg_beta_body", "spmv_dot2_body", "pcg_alpha_body",
              "k_bicg_check", "pcg_init_body"):
        assert n in found, n
    assert found["pcg_alpha_body"][0] == {"done"} and not found["pcg_alpha_body"][1]
    assert found["pcg_init_body"][1] >= {"done", "stop"}
    # the test is stored, copied and returned on somewhere
    assert any("stop" in s for _, s in found.values()) and any("stop" in r for r, _ in found.values())


def test_no_launch_stores_the_flag_it_returns_on():
    for name, body in _functions():
        reads, stores = _reads_and_stores(body)
        if name not in ONE_GROUP:
            assert not (reads & stores), f"{name} reads and stores {reads & stores}"


@pytest.mark.parametrize("body,kernels", sorted(ONE_GROUP.items()))
def test_the_others_are_launched_as_one_group(body, kernels):
    text = "".join(open(f).read() for f in glob.glob(os.path.join(CSRC, "*.h*")))
    for k in kernels:
        if k.startswith("kb_"):
            shapes = re.findall(r"launch\(" + k + r", (\w+),", text)
            assert shapes and set(shapes) == {"kShTileOne"}
            assert re.search(r"case kShTileOne: return f\.over_tiles\(\) \? 1 : 0;", text)
        else:
            grids = re.findall(r"hipLaunchKernelGGL\(" + k + r", (dim3\([^)]*\))", text)
            assert grids and set(grids) == {"dim3(1)"}
    src = dict(_functions())[body]
    store = min(m.start() for p in FLAGS.values() for m in re.finditer(p + r"\s*=(?!=)", src))
    assert re.search(r"reduce_partials|pcg_test", src[:store]), "no barrier ahead of the store"
