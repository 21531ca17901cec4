"""What a pass leaves alone and what it writes as zero.  A leaf target without refined
neighbours keeps its L_c, every leaf target its L_4..19, every slot that is no target
all of its rows; a leaf target with refined neighbours gets L_c = 0 in the cells that
no refined neighbour's cell reaches.  In a tree solve an output that is zero throughout
a node in the plain form of the kernels is zero throughout it in the form the solve
takes.  Zeros and untouched values are exact, so there is no tolerance; the written
values are compared with the oracle to 1e-12 as elsewhere.
"""
import numpy as np
import pytest

import oracle
from metrics import normwise
from octotiger_amd import _abi, hip, native, workloads
from test_gpu_p2m_lists import REFINED, as_leaf
from test_gpu_tree_levels import solve, tree_with

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize("which", ["none", "face", "corner", "few"])
@pytest.mark.parametrize("theta", [0.5, 0.34])
@pytest.mark.parametrize("type_", [_abi.RHO, _abi.DRHODT])
def test_leaf_targets_write_only_what_they_form(type_, theta, which):
    lv = workloads.uniform_level((3, 3, 3), ((1, 2),) * 3, 20261901)
    leaf = np.ones(lv.nslots, bool)
    leaf[[int(lv.neighbors[13, raw]) for raw in REFINED[which] if raw != 13]] = False
    as_leaf(lv, leaf)
    Lr, Lcr = oracle.level_interactions(lv, theta, type_)
    rng = np.random.default_rng(3)
    L0, C0 = rng.normal(size=Lr.shape) * np.abs(Lr).max(), rng.normal(size=Lcr.shape)
    ctx = native.Context(theta=theta, device=0)
    dl = hip.LevelOnDevice(lv)
    dL, dC = hip.DeviceArray.from_numpy(L0), hip.DeviceArray.from_numpy(C0)
    plan = ctx.level_plan(lv, dl.M.addr, dl.com.addr, dl.mon.addr, dL.addr, dC.addr, type_=type_)
    s = hip.Stream()
    plan.execute(s.handle)
    s.synchronize()
    L, Lc = dL.numpy(), dC.numpy()
    t = int(lv.targets[0])
    others = np.arange(lv.nslots) != t
    assert np.array_equal(L[others], L0[others]) and np.array_equal(Lc[others], C0[others])
    assert np.array_equal(L[t, :, 4:], L0[t, :, 4:])
    assert normwise(L[t, :, :4], L0[t, :, :4] + Lr[t, :, :4]) <= TOL
    if type_ == _abi.DRHODT or which == "none":
        assert np.array_equal(Lc[t], C0[t])
    else:
        alone = ~Lcr[t].any(axis=-1)
        assert alone.any() and not alone.all()
        assert not Lc[t][alone].any()
        assert normwise(Lc[t], Lcr[t]) <= TOL
    plan.close()
    for a in (dL, dC):
        a.free()
    dl.free()
    ctx.close()


@pytest.mark.parametrize("sizes", [(0, 0, 0), (1, 0, 0), (8, 3, 0), (8, 64, 96)])
@pytest.mark.parametrize("type_", [_abi.RHO, _abi.DRHODT])
def test_tree_zeros_are_those_of_the_plain_form(monkeypatch, type_, sizes):
    t = tree_with(*sizes)
    got = solve(t, 0.5, type_, 0)
    monkeypatch.setenv("OCTOFMM_VARIANT", "702")
    ref = solve(t, 0.5, type_, 0)
    zeros = 0
    for g, r in zip(got, ref):
        for k in g:
            blank = ~r[k].reshape(len(r[k]), -1).any(axis=1)
            zeros += int(blank.sum())
            assert not g[k][blank].any()
    assert zeros > 0   # refined nodes have no force rows; a lone leaf has no L_c
