"""Levels of few sub-grids, where variant 704 splits a coarse block's offsets over
several workgroups: the numbers of targets at which the number of parts changes
(most parts, a few, two, none), with leaf neighbours (near pairs), both opening
angles and both solves, against the oracle; and every split gives the plain
form's sums to rounding.

Tolerance: only the order of the sums over pairs differs, 1e-12 as elsewhere.
"""
import numpy as np
import pytest

import oracle
from metrics import normwise
from octotiger_amd import _abi, hip, native, workloads

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize("theta", [0.5, 0.34])
@pytest.mark.parametrize("n", [1, 9, 19, 29])
def test_few_targets_match_oracle(n, theta, monkeypatch):
    monkeypatch.setenv("OCTOFMM_VARIANT", "704")
    lv = workloads.uniform_level((n + 2, 3, 3), ((1, n + 1), (1, 2), (1, 2)), 20261500 + n)
    leaf = np.zeros(lv.nslots, bool)
    leaf[:9] = True                       # one end of the strip borders leaves
    lv.kind[leaf] = _abi.SLOT_LEAF
    lv.mon[leaf] = lv.M[leaf][..., 0]
    lv.M[leaf] = 0.0
    i = np.stack(np.meshgrid(*[np.arange(8.0)] * 3, indexing="ij"), -1).reshape(512, 3)
    lv.com[leaf] = (lv.xbase[:, None, :] + i * lv.dx)[leaf]
    ctx = native.Context(theta=theta, device=0)
    dl = hip.LevelOnDevice(lv)
    s = hip.Stream()
    for type_ in (_abi.RHO, _abi.DRHODT):
        Lr, Lcr = oracle.level_interactions(lv, theta, type_)
        dl.zero_outputs()
        plan = dl.plan(ctx, type_=type_)
        assert plan.stats()["variant"] == 704
        plan.execute(s.handle)
        s.synchronize()
        first = dl.L.numpy()
        assert normwise(first[lv.targets], Lr[lv.targets]) <= TOL
        if type_ == _abi.RHO:
            assert normwise(dl.L_c.numpy()[lv.targets], Lcr[lv.targets]) <= TOL
        dl.zero_outputs()
        plan.execute(s.handle)
        s.synchronize()
        assert np.array_equal(dl.L.numpy(), first)   # the same bits on every pass
        plan.close()
    dl.free()
    ctx.close()
