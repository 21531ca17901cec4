"""p2m of leaf targets from its work lists: a leaf with one refined face, edge
and corner neighbour, with all and with no refined neighbours, and a level of
leaves whose lists fill several workgroups and leave the last one ragged, at the
smallest and the largest reach of the stencil; executed twice, since cells
without a p2m pair are never written.

Tolerance: only the order of the sums over pairs differs, 1e-12 as elsewhere.
"""
import numpy as np
import pytest

import oracle
from metrics import normwise
from octotiger_amd import _abi, hip, native, workloads

pytestmark = pytest.mark.gpu

TOL = 1e-12
# raw directions (dx + 1) + 3 (dy + 1) + 9 (dz + 1)
REFINED = {"face": [12], "edge": [13 + 1 + 3], "corner": [0], "few": [4, 14, 26, 17], "all": range(27), "none": []}


def check(lv, theta, type_):
    Lr, Lcr = oracle.level_interactions(lv, theta, type_)
    ctx = native.Context(theta=theta, device=0)
    dl = hip.LevelOnDevice(lv)
    plan = ctx.level_plan(lv, dl.M.addr, dl.com.addr, dl.mon.addr, dl.L.addr, dl.L_c.addr, type_=type_)
    s = hip.Stream()
    for n in (1, 2):   # L is added to, L_c overwritten
        plan.execute(s.handle)
        s.synchronize()
        L, Lc = dl.L.numpy(), dl.L_c.numpy()
        for t in lv.targets:
            cols = 4 if lv.kind[t] == _abi.SLOT_LEAF else 20
            assert normwise(L[t, :, :cols], n * Lr[t, :, :cols]) <= TOL
            if type_ == _abi.RHO and np.abs(Lcr[t]).max() > 0.0:
                assert normwise(Lc[t], Lcr[t]) <= TOL
    plan.close()
    dl.free()
    ctx.close()


def as_leaf(lv, leaf):
    lv.kind[leaf] = _abi.SLOT_LEAF
    lv.mon[leaf] = lv.M[leaf][:, :, 0]
    lv.M[leaf] = 0.0
    i = np.stack(np.meshgrid(*[np.arange(8.0)] * 3, indexing="ij"), -1).reshape(512, 3)
    lv.com[leaf] = (lv.xbase[:, None, :] + i * lv.dx)[leaf]


@pytest.mark.parametrize("which", list(REFINED))
@pytest.mark.parametrize("theta", [0.5, 0.34])
@pytest.mark.parametrize("type_", [_abi.RHO, _abi.DRHODT])
def test_one_leaf(type_, theta, which):
    lv = workloads.uniform_level((3, 3, 3), ((1, 2),) * 3, 20261501)
    leaf = np.ones(lv.nslots, bool)
    leaf[[int(lv.neighbors[13, raw]) for raw in REFINED[which] if raw != 13]] = False
    as_leaf(lv, leaf)
    check(lv, theta, type_)


@pytest.mark.parametrize("theta", [0.5, 0.34])
@pytest.mark.parametrize("share", [0.1, 0.5])
def test_many_leaves(theta, share):
    lv = workloads.uniform_level((5, 4, 4), ((1, 4), (1, 3), (1, 3)), 20261502)
    rng = np.random.default_rng(11)
    as_leaf(lv, rng.random(lv.nslots) >= share)
    check(lv, theta, _abi.RHO)
