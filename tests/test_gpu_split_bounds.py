"""Where variant 704 stops splitting the coarse blocks of a small level over several
workgroups: the largest level it splits and the smallest it does not, at the
lengths of the far schedule, with leaf neighbours (near pairs), against the oracle
and against variant 702.  An unsplit level runs the same sums as the persistent form
804, 4 waves a block in wave order, so the two give the same bits: at theta 0.5 two
parts are slower than the plain form from 24 targets on (27.0 us against 26.3) and
must not be taken there, at theta 0.6 and 0.75 from fewer on.

Tolerance: only the order of the sums over pairs differs, 1e-12 as elsewhere.
"""
import numpy as np
import pytest

import oracle
from metrics import normwise
from octotiger_amd import _abi, hip, native, workloads

pytestmark = pytest.mark.gpu

TOL = 1e-12


def strip(n):
    """n targets in a row, one end bordering leaves."""
    lv = workloads.uniform_level((n + 2, 3, 3), ((1, n + 1), (1, 2), (1, 2)), 20261700 + n)
    leaf = np.zeros(lv.nslots, bool)
    leaf[:9] = True
    lv.kind[leaf] = _abi.SLOT_LEAF
    lv.mon[leaf] = lv.M[leaf][..., 0]
    lv.M[leaf] = 0.0
    i = np.stack(np.meshgrid(*[np.arange(8.0)] * 3, indexing="ij"), -1).reshape(512, 3)
    lv.com[leaf] = (lv.xbase[:, None, :] + i * lv.dx)[leaf]
    return lv


def one_pass(dl, ctx, s, type_):
    dl.zero_outputs()
    plan = dl.plan(ctx, type_=type_)
    variant = plan.stats()["variant"]
    plan.execute(s.handle)
    s.synchronize()
    plan.close()
    return variant, dl.L.numpy(), dl.L_c.numpy()


@pytest.mark.parametrize("theta,n,split", [
    (0.5, 22, True), (0.5, 23, False), (0.5, 28, False), (0.5, 29, False),
    (0.45, 28, True), (0.45, 29, False),
    (0.34, 36, True), (0.34, 48, True), (0.34, 49, False),
    (0.6, 18, True), (0.6, 19, False), (0.75, 16, True), (0.75, 17, False),
])
def test_split_ends_where_it_stops_paying(theta, n, split, monkeypatch):
    lv = strip(n)
    ctx = native.Context(theta=theta, device=0)
    dl = hip.LevelOnDevice(lv)
    s = hip.Stream()
    tg = lv.targets
    for type_ in (_abi.RHO, _abi.DRHODT):
        Lr, Lcr = oracle.level_interactions(lv, theta, type_)
        out = {}
        for v in (704, 804, 702):
            monkeypatch.setenv("OCTOFMM_VARIANT", str(v))
            variant, L, Lc = one_pass(dl, ctx, s, type_)
            assert variant == v
            out[v] = L[tg], Lc[tg]
        for v in (804, 702):
            assert normwise(out[704][0], out[v][0]) <= TOL
        assert normwise(out[704][0], Lr[tg]) <= TOL
        if type_ == _abi.RHO:
            assert normwise(out[704][1], Lcr[tg]) <= TOL
            assert normwise(out[704][1], out[702][1]) <= TOL
        else:
            assert not out[704][1].any()   # DRHODT leaves L_c as it was
        if not split:
            assert np.array_equal(out[704][0], out[804][0]) and np.array_equal(out[704][1], out[804][1])
    dl.free()
    ctx.close()
