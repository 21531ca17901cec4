"""Near pairs of multipole targets with leaf neighbours, whose partners are read
eight at a time: leaves at one face, edge and corner and on all sides, next to
refined and missing neighbours, with partners of either sign, for the plain and
the wide form of the kernel, against the oracle.

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
LEAVES = {"face": [14], "edge": [13 - 1 + 3], "corner": [26], "some": [4, 12, 22, 0], "all": range(27)}


@pytest.mark.parametrize("which", list(LEAVES))
@pytest.mark.parametrize("theta", [0.5, 0.34])
@pytest.mark.parametrize("type_", [_abi.RHO, _abi.DRHODT])
@pytest.mark.parametrize("variant", ["702", "704"])
def test_near_pairs(monkeypatch, variant, type_, theta, which):
    lv = workloads.uniform_level((3, 3, 3), ((1, 2),) * 3, 20261701)
    rng = np.random.default_rng(3)
    leaf = np.zeros(lv.nslots, bool)
    leaf[[int(lv.neighbors[13, raw]) for raw in LEAVES[which] if raw != 13]] = True
    if which == "some":
        lv.neighbors[13, [1, 16]] = -1
    lv.kind[leaf] = _abi.SLOT_LEAF
    lv.mon[leaf] = rng.normal(size=(int(leaf.sum()), 512))
    lv.M[leaf] = 0.0
    i = np.stack(np.meshgrid(*[np.arange(8.0)] * 3, indexing="ij"), -1).reshape(512, 3)
    lv.com[leaf] = (lv.xbase[:, None, :] + i * lv.dx)[leaf]
    Lr, Lcr = oracle.level_interactions(lv, theta, type_)
    monkeypatch.setenv("OCTOFMM_VARIANT", variant)
    ctx = native.Context(theta=theta, device=0)
    dl = hip.LevelOnDevice(lv)
    plan = ctx.level_plan(lv, dl.M.addr, dl.com.addr, dl.mon.addr, dl.L.addr, dl.L_c.addr, type_=type_)
    s = hip.Stream()
    plan.execute(s.handle)
    s.synchronize()
    L, Lc = dl.L.numpy(), dl.L_c.numpy()
    assert normwise(L[13], Lr[13]) <= TOL
    if type_ == _abi.RHO:
        assert normwise(Lc[13], Lcr[13]) <= TOL
    plan.close()
    dl.free()
    ctx.close()
