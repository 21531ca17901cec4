"""Whole-tree solves whose small levels run sums first (up to 96 targets, in one
to several workgroups per coarse block), in the launches that the coarsest levels
share or beyond them, against the plain form of the same kernels
(OCTOFMM_VARIANT), with levels of 1 to 97 targets, leaves and refined
neighbours on every side, small leaf levels that go with the next one's launch;
RHO and DRHODT, with and without a graph, with and without the leaves' rows; a
repeated solve gives the same bits.

Tolerance: the two forms differ in the order of the sums over partners only,
1e-12 as elsewhere.
"""
import numpy as np
import pytest

from metrics import normwise
from octotiger_amd import _abi, hip, native, tree as octree, workloads

pytestmark = pytest.mark.gpu

TOL = 1e-12


def tree_with(n1, n2, n3):
    """Refines n1 nodes of level 1, n2 of level 2, n3 of level 3 (before nesting)."""
    def refine(lev, cs, xb, dxl):
        want = np.zeros(len(cs), bool)
        want[: (len(cs), n1, n2, n3)[lev]] = True
        return want

    t = octree.build_tree(refine, 1 + (n1 > 0) + (n2 > 0) + (n3 > 0), name="levels")
    workloads._assign_leaf_masses(t, lambda x: np.ones(x.shape[:-1]), 20261601, 1.0)
    return t


def solve(t, theta, type_, flags):
    ctx = native.Context(theta=theta, device=0)
    dev = hip.TreeOnDevice(t)
    s = hip.Stream()
    out = []
    for ty in ((_abi.RHO,) if type_ == _abi.RHO else (_abi.RHO, _abi.DRHODT)):
        plan = dev.plan(ctx, type_=ty, flags=flags)
        for _ in range(2):
            plan.execute(s.handle)
            s.synchronize()
            out.append(dev.fetch("L", "L_c", "g"))
        plan.close()
    dev.free()
    ctx.close()
    for a, b in zip(*out[-2:]):
        for k in a:
            assert np.array_equal(a[k], b[k])
    return out[-1]


def compare(monkeypatch, t, theta, type_, flags):
    print([int((lv.kind == _abi.SLOT_NONLEAF).sum()) for lv in t.levels], flush=True)
    got = solve(t, theta, type_, flags)
    monkeypatch.setenv("OCTOFMM_VARIANT", "702")
    ref = solve(t, theta, type_, flags)
    for g, r in zip(got, ref):
        for k in g:
            assert np.isfinite(g[k]).all()
            if np.abs(r[k]).max() > 0.0:
                assert normwise(g[k], r[k]) <= TOL


@pytest.mark.parametrize("sizes", [(0, 0, 0), (1, 0, 0), (8, 3, 0), (8, 64, 96), (8, 64, 97)])
@pytest.mark.parametrize("theta", [0.5, 0.34])
@pytest.mark.parametrize("type_", [_abi.RHO, _abi.DRHODT])
def test_sums_first_matches_plain(monkeypatch, type_, theta, sizes):
    flags = _abi.PLAN_USE_GRAPH if sizes[1] else 0
    if sizes[0] == 1:
        flags |= _abi.TREE_LEAF_G_ONLY
    compare(monkeypatch, tree_with(*sizes), theta, type_, flags)


def test_small_leaf_level_after_large_ones(monkeypatch):
    t = tree_with(8, 64, 280)
    leaves = [int((lv.kind == _abi.SLOT_LEAF).sum()) for lv in t.levels]
    assert sum(lv.nnodes for lv in t.levels[:4]) > 256 and 0 < leaves[3] <= 256 < leaves[4]
    compare(monkeypatch, t, 0.5, _abi.RHO, _abi.PLAN_USE_GRAPH)
