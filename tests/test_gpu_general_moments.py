"""GPU parity on general moments: the level and leaf kernels contract trace-free
parts of the quadrupoles and octupoles and put the traces back by identities of
the harmonic derivatives, so moments with large traces, dipoles and either sign
(which masses about their centre of mass never have) go against the oracle,
per component normwise.

Tolerance: a pair's terms carry at most 7 times the reciprocal root's 4.1e-15
plus a few roundings, 4e-14 of the terms; the random signs of the moments leave
a component's largest sum no smaller than its largest term: 1e-12 as elsewhere.
"""
import numpy as np
import pytest

import oracle
from metrics import normwise
from octotiger_amd import _abi, hip, native, workloads

pytestmark = pytest.mark.gpu

TOL = 1e-12


def general_level(kinds, seed=20261301):
    """3 x 3 x 3 slots, the centre and one neighbour targets, with random
    moments of the size mass dx^order and centres anywhere in the cell."""
    lv = workloads.uniform_level((4, 3, 3), ((1, 3), (1, 2), (1, 2)), seed)
    rng = np.random.default_rng(seed)
    order = np.array([0] + [1] * 3 + [2] * 6 + [3] * 10)
    M = rng.normal(size=lv.M.shape) * lv.dx ** order
    M[..., [4, 7, 9]] += 3.0 * lv.dx ** 2                 # a trace larger than the rest
    M[..., 10] += 2.0 * lv.dx ** 3
    M[..., 0] = np.where(rng.random(M.shape[:2]) < 0.5, -1.0, 1.0) * rng.uniform(0.5, 2.0, M.shape[:2])
    lv.M[:] = M
    if kinds == "mixed":
        leaf = rng.random(lv.nslots) < 0.5
        leaf[lv.targets] = [True, False]
        lv.kind[leaf] = _abi.SLOT_LEAF
        lv.mon[leaf] = rng.normal(size=(int(leaf.sum()), 512))
        lv.M[leaf] = 0.0
        i = np.stack(np.meshgrid(*[np.arange(8.0)] * 3, indexing="ij"), -1).reshape(512, 3)
        lv.com[leaf] = (lv.xbase[:, None, :] + i * lv.dx)[leaf]
    return lv


@pytest.mark.parametrize("theta", [0.5, 0.34])
@pytest.mark.parametrize("kinds", ["refined", "mixed"])
@pytest.mark.parametrize("type_", [_abi.RHO, _abi.DRHODT])
def test_general_moments_match_oracle(type_, kinds, theta):
    lv = general_level(kinds)
    Lr, Lcr = oracle.level_interactions(lv, theta, type_)
    ctx = native.Context(theta=theta, device=0)
    dl = hip.LevelOnDevice(lv)
    s = hip.Stream()
    for variant in (_abi.PLAN_USE_GRAPH, _abi.PLAN_USE_GRAPH | _abi.PLAN_AUTOTUNE):
        dl.zero_outputs()
        plan = dl.plan(ctx, type_=type_, flags=variant)
        plan.execute(s.handle)
        s.synchronize()
        L, Lc = dl.L.numpy(), dl.L_c.numpy()
        for t in lv.targets:
            rows = 4 if lv.kind[t] == _abi.SLOT_LEAF else 20
            assert normwise(L[t, :, :rows], Lr[t, :, :rows]) <= TOL
            if type_ == _abi.RHO:
                assert normwise(Lc[t], Lcr[t]) <= TOL
        plan.close()
    dl.free()
    ctx.close()


@pytest.mark.parametrize("type_", [_abi.RHO, _abi.DRHODT])
def test_general_moments_root(type_):
    lv = general_level("refined")
    sg, keep = workloads.subgrid_view(lv, int(lv.targets[0]), root=True, type_=type_)
    Lr, Lcr = oracle.multipole_interactions(sg)
    ctx = native.Context(theta=0.5, device=0)
    L, Lc = np.zeros((512, 20)), np.zeros((512, 3))
    ctx.multipole_interactions(sg, L, Lc)
    ctx.close()
    assert normwise(L, Lr) <= TOL
    if type_ == _abi.RHO:
        assert normwise(Lc, Lcr) <= TOL
