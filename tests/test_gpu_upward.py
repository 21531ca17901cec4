"""The upward pass over leaves, one wave per leaf and four to a workgroup:
multipoles and centres of mass of the cells above, and the leaf cells' centres,
against moments summed in extended precision, for leaf counts that leave the
last workgroup ragged, a tree that is a single leaf, masses and centres at
addresses that are only 8-byte aligned, and (DRHODT) sources of either sign
about given centres.

Tolerance: each moment against the size of its terms, sum |m| dx^order, 1e-12 as
elsewhere; the geometric centres of the leaf cells are exact.
"""
import numpy as np
import pytest

from octotiger_amd import _abi, hip, native, tree as octree, workloads

pytestmark = pytest.mark.gpu

TOL = 1e-12
PAIRS = [(a, b) for a in range(3) for b in range(a, 3)]
TRIPLES = [(a, b, c) for a in range(3) for b in range(a, 3) for c in range(b, 3)]


def moments(m, X, Y):
    """[..., 8] masses at [..., 8, 3] about [..., 3]: 20 components."""
    d = (X - Y[..., None, :]).astype(np.longdouble)
    m = m.astype(np.longdouble)
    out = [m.sum(-1)] + [(m * d[..., a]).sum(-1) for a in range(3)]
    out += [(m * d[..., a] * d[..., b]).sum(-1) for a, b in PAIRS]
    out += [(m * d[..., a] * d[..., b] * d[..., c]).sum(-1) for a, b, c in TRIPLES]
    return np.stack(out, -1)


def coarse(a):
    """[512, ...] cells -> [4, 4, 4, 8, ...] children of each coarse cell."""
    t = a.shape[1:]
    return a.reshape((4, 2, 4, 2, 4, 2) + t).transpose((0, 2, 4, 1, 3, 5) + tuple(range(6, 6 + len(t)))).reshape((4, 4, 4, 8) + t)


@pytest.mark.parametrize("refined", [None, 0, 1, 3, 7])
@pytest.mark.parametrize("type_", [_abi.RHO, _abi.DRHODT])
def test_leaf_moments(type_, refined):
    def refine(lev, cs, xb, dxl):
        return np.arange(len(cs)) < (len(cs) if lev == 0 else refined)

    t = octree.build_tree(refine, 0 if refined is None else 1 + (refined > 0), lo=-0.3, size=1.7, name="upward")
    workloads._assign_leaf_masses(t, lambda x: np.ones(x.shape[:-1]), 20261801, 1.0)
    rng = np.random.default_rng(5)
    ctx = native.Context(theta=0.5, device=0)
    dev = hip.TreeOnDevice(t)
    odd, addr = [], dev.addresses()
    given = []
    for lv, d, a in zip(t.levels, dev.levels, addr):
        mon = lv.mon if type_ == _abi.RHO else rng.normal(size=(lv.nnodes, 512))
        com = t.cell_centres(lv) + rng.uniform(-0.3, 0.3, size=(lv.nnodes, 512, 3)) * lv.dx
        given.append((mon, com))
        for k, v in (("mon", mon), ("com", com)):
            odd.append(hip.DeviceArray.from_numpy(np.concatenate([[0.0], np.ascontiguousarray(v).reshape(-1)])))
            a[k] = odd[-1].addr + 8
    plan = ctx.tree_plan(t, addr, type_=type_)
    s = hip.Stream()
    plan.execute(s.handle)
    s.synchronize()
    com = [odd[2 * i + 1].numpy()[1:].reshape(lv.nnodes, 512, 3) for i, lv in enumerate(t.levels)]
    M = [d["M"].numpy() for d in dev.levels]
    order = np.array([0] + [1] * 3 + [2] * 6 + [3] * 10)
    for l, lv in enumerate(t.levels):
        leaf = np.nonzero(lv.kind == _abi.SLOT_LEAF)[0]
        X = t.cell_centres(lv) if type_ == _abi.RHO else given[l][1]
        assert np.array_equal(com[l][leaf], X[leaf])
        if l == 0:
            continue
        for n in leaf:
            p, o = int(lv.parent[n]), int(lv.octant[n])
            at = np.s_[4 * (o & 1):4 * (o & 1) + 4, 4 * (o >> 1 & 1):4 * (o >> 1 & 1) + 4, 4 * (o >> 2):4 * (o >> 2) + 4]
            Y = com[l - 1][p].reshape(8, 8, 8, 3)[at]
            m, x = coarse(given[l][0][n]), coarse(X[n])
            if type_ == _abi.RHO:
                ref = (m.astype(np.longdouble)[..., None] * x).sum(-2) / m.astype(np.longdouble).sum(-1)[..., None]
                assert np.abs(Y - ref).max() <= TOL * t.size
            got = M[l - 1][p].reshape(8, 8, 8, 20)[at]
            scale = np.abs(m).sum(-1)[..., None] * lv.dx ** order
            assert (np.abs(got - moments(m, x, Y)) <= TOL * scale).all()
    plan.close()
    for a in odd:
        a.free()
    dev.free()
    ctx.close()
