"""p2p of leaf targets at theta = 0.5, where opposite partners are folded before
they meet their constants: every child class of the window's edges against the
oracle, over neighbourhoods with leaf, refined and missing slots, with signed
monopoles (so no sum of opposite cells is small by itself) and with the
monopoles at an address that is only 8-byte aligned.

Tolerance: 215 partners of either sign, each product rounded a few times at
1.1e-16, against a component's largest sum: 1e-12 as elsewhere.
"""
import numpy as np
import pytest

import oracle
from metrics import normwise
from octotiger_amd import _abi, hip, native, workloads

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize("pattern", ["leaves", "kinds", "edge"])
@pytest.mark.parametrize("type_", [_abi.RHO, _abi.DRHODT])
def test_folded_p2p_matches_oracle(type_, pattern):
    lv = workloads.uniform_level((4, 3, 3), ((1, 3), (1, 2), (1, 2)), 20261401)
    rng = np.random.default_rng(7)
    leaf = np.ones(lv.nslots, bool) if pattern == "leaves" else rng.random(lv.nslots) < 0.6
    leaf[lv.targets] = True
    if pattern == "edge":   # missing directions, as at a domain boundary
        gone = rng.random(lv.nslots) < 0.5
        gone[lv.targets] = False
        lv.neighbors[np.isin(lv.neighbors, np.nonzero(gone)[0])] = -1
        lv.neighbors[:, 13] = np.arange(lv.nslots)
    lv.kind[leaf] = _abi.SLOT_LEAF
    lv.mon[leaf] = rng.normal(size=(int(leaf.sum()), 512))
    lv.M[leaf] = 0.0
    i = np.stack(np.meshgrid(*[np.arange(8.0)] * 3, indexing="ij"), -1).reshape(512, 3)
    lv.com[leaf] = (lv.xbase[:, None, :] + i * lv.dx)[leaf]
    Lr, Lcr = oracle.level_interactions(lv, 0.5, type_)
    ctx = native.Context(theta=0.5, device=0)
    dl = hip.LevelOnDevice(lv)
    odd = hip.DeviceArray.from_numpy(np.concatenate([[0.0], lv.mon.reshape(-1)]))
    plan = ctx.level_plan(lv, dl.M.addr, dl.com.addr, odd.addr + 8, dl.L.addr, dl.L_c.addr, type_=type_)
    s = hip.Stream()
    plan.execute(s.handle)
    s.synchronize()
    L, Lc = dl.L.numpy(), dl.L_c.numpy()
    for t in lv.targets:
        assert normwise(L[t, :, :4], Lr[t, :, :4]) <= TOL
        if type_ == _abi.RHO and np.abs(Lcr[t]).max() > 0.0:
            assert normwise(Lc[t], Lcr[t]) <= TOL
    plan.close()
    odd.free()
    dl.free()
    ctx.close()
