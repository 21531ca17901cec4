"""The gravity work a user of this framework has it do, as cases to time.

Three families, each through the entry point a program calls:

  dropin  one sub-grid with its 26 neighbours in host memory, through
          Context.multipole_interactions / monopole_interactions (the
          per-node calls an unmodified Octo-Tiger makes);
  level   every sub-grid of one octree level in device memory, through a level
          plan (Context.level_plan, one graph per pass, autotuned);
  tree    a whole adaptive-tree solve in device memory, through a tree plan
          (Context.tree_plan: M2M, interactions of every level, L2L, forces).

A case is a dict of plain values; prepare() makes its inputs on the GPU (host
memory for dropin) from the seed alone and creates the plan, run() is one pass,
exact() the same outputs in plain 64-bit torch, without this package's code.
"""
import functools
import math

import numpy as np
import torch

from octotiger_amd import _abi, native, workloads

CELLS = 512
TYPES = {"rho": _abi.RHO, "drhodt": _abi.DRHODT}
FLAGS = _abi.PLAN_USE_GRAPH | _abi.PLAN_AUTOTUNE
# nominal operations of one pair in the reference's source (fused multiply-add = 2)
FLOPS = {"rho": {"m2l": 407, "p2m": 318, "p2p": 12}, "drhodt": {"m2l": 273, "p2m": 205, "p2p": 12}}
SPHERE, POLYTROPE_THRESHOLD = "sphere", 2.5e-8


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def _dropin(entry, type_="rho", refined=26, leaves=0, theta=0.5):
    return {"family": "dropin", "entry": entry, "type": type_, "refined": refined, "leaves": leaves, "theta": theta}


def _level(nx, ny, nz, type_="rho", precision="fp64", leaf_fraction=0.0, theta=0.5, partial=False):
    return {"family": "level", "nx": nx, "ny": ny, "nz": nz, "type": type_, "precision": precision,
            "leaf_fraction": leaf_fraction, "theta": theta, "partial": partial}


def _tree(shape, max_level, threshold, type_="rho", leaf_g_only=False):
    return {"family": "tree", "shape": shape, "max_level": max_level, "threshold": threshold, "type": type_,
            "leaf_g_only": leaf_g_only}


def listed():
    return [
        # one refined node of an Octo-Tiger run, all neighbours refined: the per-node drop-in call
        dict(_dropin("nonleaf"), name="dropin-nonleaf"),
        # one leaf at a refinement boundary: p2p with 17 leaf neighbours, p2m with 9 refined ones
        dict(_dropin("leaf", refined=9, leaves=17), name="dropin-leaf"),
        # a coarse level of a tree, or one rank's share of a level: few sub-grids, ragged box
        dict(_level(5, 3, 3), name="level-45-ragged"),
        # a mid-size level (the 512-sub-grid benchmark level)
        dict(_level(8, 8, 8), name="level-512"),
        # the headline level of the benchmark: 4096 sub-grids, RHO with the angular-momentum correction
        dict(_level(16, 16, 16), name="level-4096"),
        # the other solve of every production step, on the same level
        dict(_level(16, 16, 16, type_="drhodt"), name="level-4096-drhodt"),
        # the mixed-precision option on the same level
        dict(_level(16, 16, 16, precision="mixed"), name="level-4096-mixed"),
        # a level of mixed refinement: near pairs, p2p and p2m beside M2L (the 2048-sub-grid benchmark level)
        dict(_level(16, 16, 8, leaf_fraction=0.4), name="level-2048-kinds"),
        # the smallest opening angle (about five times the pairs per cell), halo slots handed over
        # partially as remote neighbours hand them over, ragged box with some leaves
        dict(_level(7, 5, 3, leaf_fraction=0.2, theta=0.34, partial=True), name="level-105-theta034"),
        # Octo-Tiger's solid-sphere regression tree (329 sub-grids): a small solve, bound by latency
        dict(_tree(SPHERE, 3, 0.0), name="tree-329-sphere"),
        # the production solve of a polytrope (10,697 sub-grids on levels 0..6), both halves of a step
        dict(_tree("polytrope", 6, POLYTROPE_THRESHOLD), name="tree-10697"),
        dict(_tree("polytrope", 6, POLYTROPE_THRESHOLD, type_="drhodt"), name="tree-10697-drhodt"),
    ]


def draw(rng):
    family = rng.choice(["dropin", "level", "level", "level", "tree"])
    type_ = rng.choice(["rho", "rho", "drhodt"])
    if family == "dropin":
        entry = rng.choice(["nonleaf", "leaf", "root"])
        if entry == "root":
            return _dropin(entry, type_, 0, 0, round(rng.uniform(0.34, 0.5), 3))
        refined = rng.randint(3, 26) if entry == "nonleaf" else rng.randint(0, 20)
        return _dropin(entry, type_, refined, rng.randint(0, 26 - refined), rng.choice([0.34, 0.45, 0.5, 0.5]))
    if family == "level":
        theta = rng.choice([0.34, 0.45, 0.5, 0.5, 0.5])
        # sub-grids from a handful to the 4096 of the benchmark level (0.34 has up to six times the pairs)
        n = math.exp(rng.uniform(math.log(4), math.log(4096 if theta == 0.5 else 600)))
        nx = max(1, min(40, round(n ** (1 / 3) * math.exp(rng.uniform(-0.4, 0.4)))))
        ny = max(1, min(40, round(math.sqrt(n / nx) * math.exp(rng.uniform(-0.3, 0.3)))))
        nz = max(1, min(40, int(n / (nx * ny))))
        # mixed precision is for levels that fill the GPU
        mixed = theta == 0.5 and nx * ny * nz >= 512 and rng.random() < 0.3
        frac = 0.0 if mixed else rng.choice([0.0, 0.0, round(rng.uniform(0.1, 0.9), 2)])
        return _level(nx, ny, nz, type_, "mixed" if mixed else "fp64", frac, theta, rng.random() < 0.3)
    if rng.random() < 0.15:
        return _tree(SPHERE, 3, 0.0, "drhodt", False)
    # from a few dozen sub-grids to about ten thousand
    lev = rng.choice([2, 3, 4, 5, 6])
    thr = POLYTROPE_THRESHOLD * 8.0 ** (6 - lev) * math.exp(rng.uniform(0.0, 0.9))
    return _tree("polytrope", lev, float("%.3g" % thr), type_, type_ == "rho" and rng.random() < 0.3)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _rng(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _unit_cells(dev):
    i = torch.arange(CELLS, device=dev)
    return torch.stack([i // 64, (i // 8) % 8, i % 8], dim=1).to(torch.float64)


def _moments(mass_of, centre, dx, gen):
    """(M [n,512,20], com [n,512,3]) of cells that hold 8 point masses at their
    child centres, log-normal (sigma = mass_of's) about a density."""
    dev = centre.device
    off = torch.tensor([[(c >> 2) & 1, (c >> 1) & 1, c & 1] for c in range(8)], dtype=torch.float64, device=dev) - 0.5
    pos = centre[:, :, None, :] + off * (0.5 * dx)
    sigma, density = mass_of
    m = torch.exp(sigma * torch.randn(pos.shape[:3], generator=gen, dtype=torch.float64, device=dev)) * (0.5 * dx) ** 3
    if density is not None:
        m = m * density(pos)
    mass = m.sum(2)
    com = (m[..., None] * pos).sum(2) / mass[..., None]
    r = pos - com[:, :, None, :]
    M = torch.empty(mass.shape + (20,), dtype=torch.float64, device=dev)
    M[..., 0] = mass
    for a in range(3):
        ma = m * r[..., a]
        M[..., 1 + a] = ma.sum(2)
        for b in range(a, 3):
            mab = ma * r[..., b]
            M[..., _I2[a][b]] = mab.sum(2)
            for c in range(b, 3):
                M[..., _I3[a][b][c]] = (mab * r[..., c]).sum(2)
    return M, com


@functools.lru_cache(maxsize=None)
def _box(nx, ny, nz):
    """Neighbour table, slot coordinates and targets of an nx x ny x nz block
    of sub-grids inside a one-slot halo shell."""
    s = (nx + 2, ny + 2, nz + 2)
    c = np.stack(np.meshgrid(*[np.arange(v) for v in s], indexing="ij"), -1).reshape(-1, 3)
    nb = np.empty((len(c), 27), np.int32)
    for raw in range(27):
        q = c + np.array([raw % 3 - 1, raw // 3 % 3 - 1, raw // 9 - 1])
        ok = ((q >= 0) & (q < np.array(s))).all(1)
        nb[:, raw] = np.where(ok, (q[:, 0] * s[1] + q[:, 1]) * s[2] + q[:, 2], -1)
    inner = ((c > 0) & (c < np.array(s) - 1)).all(1)
    return nb, c, np.nonzero(inner)[0].astype(np.int32)


def _level_shape(case):
    """(neighbours, kind, xbase, dx, targets, coordinates): leaves are the
    slots farthest from the block's centre, as around a star."""
    nb, c, tg = _box(case["nx"], case["ny"], case["nz"])
    dx = 1.0 / (8 * (max(case["nx"], case["ny"], case["nz"]) + 2))
    xbase = (8.0 * c + 0.5) * dx
    kind = np.full(len(c), _abi.SLOT_NONLEAF, np.int32)
    nleaf = int(round(case["leaf_fraction"] * len(tg)))
    if nleaf:
        wobble = 1.0 + 0.05 * np.sin(12.9898 * c[:, 0] + 78.233 * c[:, 1] + 37.719 * c[:, 2])
        r = np.sqrt(((c - c.mean(0)) ** 2).sum(1)) * wobble
        kind[r >= np.sort(r[tg])[::-1][nleaf - 1]] = _abi.SLOT_LEAF
    return nb, kind, xbase, dx, tg, c


def _level_state(case, seed):
    """Device arrays M, com, mon of a level (zeros where a kind holds none)."""
    nb, kind, xbase, dx, tg, c = _level_shape(case)
    dev, gen = _device(), _rng(seed)
    centre = torch.as_tensor(xbase, device=dev)[:, None, :] + _unit_cells(dev) * dx
    if case["leaf_fraction"] > 0:
        mid = centre.reshape(-1, 3).mean(0)
        # a softened r^-3 profile with 5% noise, as around a star
        mass_of = (0.05, lambda p: (1.0 + ((p - mid) ** 2).sum(-1) / 0.01) ** -1.5)
    else:
        mass_of = (1.0, None)
    n = len(kind)
    M = torch.zeros(n, CELLS, 20, dtype=torch.float64, device=dev)
    com = centre.clone()
    mon = torch.zeros(n, CELLS, dtype=torch.float64, device=dev)
    leaf = torch.as_tensor(kind == _abi.SLOT_LEAF, device=dev)
    for i in range(0, n, 1024):
        Mi, ci = _moments(mass_of, centre[i:i + 1024], dx, gen)
        if case["type"] == "drhodt":
            # rates of change: signed sources about the centres of mass of the last solve
            sign = torch.randn(Mi.shape[:2], generator=gen, dtype=torch.float64, device=dev)
            Mi = Mi * sign[..., None]
        lf = leaf[i:i + 1024]
        mon[i:i + 1024] = torch.where(lf[:, None], Mi[..., 0], 0.0)
        M[i:i + 1024] = torch.where(lf[:, None, None], 0.0, Mi)
        com[i:i + 1024] = torch.where(lf[:, None, None], centre[i:i + 1024], ci)
    return M, com, mon


def _halo_cells(case):
    """{slot: cells} of the halo slots, each with the cells within 4 of the
    block: what a remote neighbour hands over."""
    nb, kind, xbase, dx, tg, c = _level_shape(case)
    size = np.array([case["nx"], case["ny"], case["nz"]]) + 1
    cell = np.stack([np.arange(CELLS) // 64, np.arange(CELLS) // 8 % 8, np.arange(CELLS) % 8], 1)
    out = {}
    for s in np.nonzero(((c == 0) | (c == size)).any(1))[0]:
        keep = ((c[s] != 0) | (cell >= 4)) & ((c[s] != size) | (cell < 4))
        out[int(s)] = np.nonzero(keep.all(1))[0].astype(np.int32)
    return out


def _dropin_level(case, seed):
    """The 27 slots around one sub-grid, as a level of one target: the first
    `refined` directions hold refined neighbours, the next `leaves` leaves, the
    rest lie outside the domain."""
    root = case["entry"] == "root"
    lv = _level(1, 1, 1, case["type"], theta=case["theta"])
    M, com, mon = (a.cpu().numpy() for a in _level_state(lv, seed))
    nb, kind, xbase, dx, tg, c = _level_shape(lv)
    nb, kind = nb.copy(), kind.copy()
    order = np.array([nb[13, r] for r in range(27) if r != 13])
    order = order[np.random.default_rng(20261202).permutation(26)]
    cell = _unit_cells(torch.device("cpu")).numpy()
    for s in list(order[case["refined"]:case["refined"] + case["leaves"]]) + [13] * (case["entry"] == "leaf"):
        kind[s] = _abi.SLOT_LEAF
        mon[s], M[s] = M[s][:, 0], 0.0
        com[s] = xbase[s] + cell * dx
    gone = order[0 if root else case["refined"] + case["leaves"]:]
    nb[np.isin(nb, gone)] = -1
    return workloads.Level("dropin", dx, (3, 3, 3), nb, kind, xbase, tg, M, com, mon)


@functools.lru_cache(maxsize=None)
def _tree_shape(shape, max_level, threshold):
    if shape == SPHERE:
        return workloads.solid_sphere_tree(max_level)
    return workloads.polytrope_tree(max_level=max_level, mass_threshold=threshold, noise_sigma=0.0)


@functools.lru_cache(maxsize=None)
def _leaf_masses(shape, max_level, threshold, level):
    return torch.as_tensor(_tree_shape(shape, max_level, threshold).levels[level].mon, device=_device())


def _tree_masses(case, seed):
    """Per level the leaf masses (1% log-normal noise) and, for DRHODT, their
    signed rates of change."""
    gen, key = _rng(seed), (case["shape"], case["max_level"], case["threshold"])
    mass, rate = [], []
    for i in range(len(_tree_shape(*key).levels)):
        base = _leaf_masses(*key, i)
        z = torch.randn(base.shape, generator=gen, dtype=torch.float64, device=base.device)
        mass.append(base * torch.exp(0.01 * z))
        rate.append(base * torch.randn(base.shape, generator=gen, dtype=torch.float64, device=base.device))
    return mass, rate


# ---------------------------------------------------------------------------
# Passes
# ---------------------------------------------------------------------------
def prepare(case, seed):
    ctx = native.Context(theta=case.get("theta", 0.5), device=0)
    type_ = TYPES[case["type"]]
    if case["family"] == "dropin":
        lv = _dropin_level(case, seed)
        sg, keep = workloads.subgrid_view(lv, 13, root=case["entry"] == "root", type_=type_)
        return {"family": "dropin", "entry": case["entry"], "ctx": ctx, "sg": sg, "keep": keep,
                "p2m": case["refined"] > 0, "L": np.zeros((CELLS, 20)), "L_c": np.zeros((CELLS, 3))}
    dev = _device()

    def zeros(n, *row):
        return torch.zeros((n, CELLS) + row, dtype=torch.float64, device=dev)

    if case["family"] == "level":
        nb, kind, xbase, dx, tg, c = _level_shape(case)
        M, com, mon = _level_state(case, seed)
        n = len(kind)
        out = {"L": zeros(n, 20), "L_c": zeros(n, 3)}
        partial, keep = None, [M, com, mon]
        if case["partial"]:
            partial = []
            for s, cells in _halo_cells(case).items():
                at = torch.as_tensor(cells, device=dev).long()
                d = {"slot": s, "cells": cells}
                for k, a in (("M", M), ("com", com)) if kind[s] == _abi.SLOT_NONLEAF else (("mon", mon),):
                    keep.append(a[s, at].contiguous())
                    d[k] = keep[-1].data_ptr()
                partial.append(d)
        torch.cuda.synchronize()
        shape = workloads.Level("level", dx, (), nb, kind, xbase, tg, None, None, None)
        plan = ctx.level_plan(shape, M.data_ptr(), com.data_ptr(), mon.data_ptr(), out["L"].data_ptr(),
                              out["L_c"].data_ptr(), type_=type_, flags=FLAGS, partial=partial,
                              precision=_abi.PRECISION_MIXED if case["precision"] == "mixed" else _abi.PRECISION_FP64)
        return {"family": "level", "ctx": ctx, "plan": plan, "keep": keep, "out": out}

    tree = _tree_shape(case["shape"], case["max_level"], case["threshold"])
    mass, rate = _tree_masses(case, seed)
    bufs = [{"M": zeros(lv.nnodes, 20), "com": zeros(lv.nnodes, 3), "mon": m, "L": zeros(lv.nnodes, 20),
             "L_c": zeros(lv.nnodes, 3), "g": zeros(lv.nnodes, 4)} for lv, m in zip(tree.levels, mass)]
    torch.cuda.synchronize()

    def plan_of(t, flags):
        return ctx.tree_plan(tree, [{k: v.data_ptr() for k, v in b.items()} for b in bufs], type_=t, flags=flags)

    if case["type"] == "drhodt":
        # the centres of mass come from the RHO solve before
        last = plan_of(_abi.RHO, 0)
        last.execute(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        last.close()
        for b, r in zip(bufs, rate):
            b["mon"] = r
            for k in ("M", "L", "L_c", "g"):
                b[k].zero_()
        torch.cuda.synchronize()
    plan = plan_of(type_, FLAGS | (_abi.TREE_LEAF_G_ONLY if case["leaf_g_only"] else 0))
    keys = ("M", "com", "L", "L_c", "g") if case["type"] == "rho" else ("M", "L", "g")
    return {"family": "tree", "ctx": ctx, "plan": plan, "bufs": bufs,
            "out": [{k: b[k] for k in keys} for b in bufs]}


def run(state):
    if state["family"] == "dropin":
        if state["entry"] == "leaf":
            state["ctx"].monopole_interactions(state["sg"], state["p2m"], state["L"], state["L_c"])
        else:
            state["ctx"].multipole_interactions(state["sg"], state["L"], state["L_c"])
        return {"L": state["L"], "L_c": state["L_c"]}
    state["plan"].execute(torch.cuda.current_stream().cuda_stream)
    return state["out"]


# ---------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _stencil(theta):
    """[(coarse offset, far [8 classes, 8 children], near)] of the opening
    criterion: coarse distance below 1 / theta, far where the fine distance
    reaches it."""
    out = []
    for d in np.ndindex(5, 5, 5):
        d = np.array(d) - 2
        if not float((d * d).sum()) < (1.0 / theta) * (1.0 / theta):
            continue
        k = np.array([[(i >> 2) & 1, (i >> 1) & 1, i & 1] for i in range(8)])
        f2 = ((2 * d + k[None, :, :] - k[:, None, :]) ** 2).sum(-1)
        far = (f2 > 0) & (1.0 / np.sqrt(np.maximum(f2, 1e-20)) <= theta)
        out.append((tuple(int(v) for v in d), far, (f2 > 0) & ~far))
    return out


def _coarse_step(delta):
    """Direction (raw) and coarse index reached from the 64 coarse cells."""
    p = np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), -1).reshape(-1, 3) + np.array(delta)
    side = np.where(p < 0, 0, np.where(p < 4, 1, 2))
    return side[:, 0] + 3 * side[:, 1] + 9 * side[:, 2], (p & 3) @ np.array([16, 4, 1])


def _level_work(nb, kind, tg, theta, type_):
    """Pairs by kind of one level pass, as (flops, bytes)."""
    far, near = np.zeros(27), np.zeros(27)
    for delta, f, n in _stencil(theta):
        raw, _ = _coarse_step(delta)
        np.add.at(far, raw, f.sum())
        np.add.at(near, raw, n.sum())
    nbk = np.where(nb[tg] >= 0, kind[np.maximum(nb[tg], 0)], -1)
    is_leaf = kind[tg] == _abi.SLOT_LEAF
    leaf_nb, ref_nb = nbk == _abi.SLOT_LEAF, nbk == _abi.SLOT_NONLEAF
    m2l = ((leaf_nb | ref_nb)[~is_leaf] @ far).sum() + (leaf_nb[~is_leaf] @ near).sum()
    p2p = (leaf_nb[is_leaf] @ (far + near)).sum()
    p2m = (ref_nb[is_leaf] @ (far + near)).sum()
    w = FLOPS[type_]
    flops = m2l * w["m2l"] + p2p * w["p2p"] + p2m * w["p2m"]
    used = np.unique(np.concatenate([nb[tg][nb[tg] >= 0], tg]))
    used_leaf = int((kind[used] == _abi.SLOT_LEAF).sum())
    row = 20 * 2 + (3 if type_ == "rho" else 0)
    leaf_row = 4 * 2 + (3 if type_ == "rho" else 0)
    words = 23 * (len(used) - used_leaf) + used_leaf + row * int((~is_leaf).sum()) + leaf_row * int(is_leaf.sum())
    return float(flops), 8.0 * CELLS * words


def work(case):
    if case["family"] == "dropin":
        n = 1 + case["refined"] + case["leaves"]
        nb = np.full((27, 27), -1, np.int32)
        nb[13, :13], nb[13, 14:] = np.arange(13), np.arange(14, 27)
        nb[13, 13] = 13
        order = np.array([r for r in range(27) if r != 13])[np.random.default_rng(20261202).permutation(26)]
        kind = np.full(27, _abi.SLOT_NONLEAF, np.int32)
        kind[order[case["refined"]:n - 1]] = _abi.SLOT_LEAF
        kind[13] = _abi.SLOT_LEAF if case["entry"] == "leaf" else _abi.SLOT_NONLEAF
        nb[13, order[n - 1:]] = -1
        flops, size = _level_work(nb, kind, np.array([13]), case["theta"], case["type"])
        if case["entry"] == "root":
            flops = 251496.0 * FLOPS[case["type"]]["m2l"]
        return {"flops": flops, "bytes": size}
    if case["family"] == "level":
        nb, kind, xbase, dx, tg, c = _level_shape(case)
        flops, size = _level_work(nb, kind, tg, case["theta"], case["type"])
        return {"flops": flops, "bytes": size}
    flops, words = 251496.0 * FLOPS[case["type"]]["m2l"], 0
    for i, lv in enumerate(_tree_shape(case["shape"], case["max_level"], case["threshold"]).levels):
        if i > 0:
            flops += _level_work(lv.neighbors, lv.kind, np.arange(lv.nnodes), 0.5, case["type"])[0]
        rho = case["type"] == "rho"
        # non-leaf: M and (RHO) com written, L and L_c written; leaf: mon read, com, L, L_c and g written
        words += (lv.nnodes - lv.nleaves) * (40 + 6 * rho)
        words += lv.nleaves * (1 + (0 if case["leaf_g_only"] else 20) + (10 if rho else 1))
    return {"flops": flops, "bytes": 8.0 * CELLS * words}


# ---------------------------------------------------------------------------
# The same outputs in plain 64-bit torch
# ---------------------------------------------------------------------------
_I2 = [[4, 5, 6], [5, 7, 8], [6, 8, 9]]
_I3 = [[[10, 11, 12], [11, 13, 14], [12, 14, 15]], [[11, 13, 14], [13, 16, 17], [14, 17, 18]],
       [[12, 14, 15], [14, 17, 18], [15, 18, 19]]]
_R3 = range(3)


def _pair_sums(x, m, ratio, octupole, dipole, rows):
    """Expansion rows [rows] and correction [3] of pairs at separations x
    (lists of tensors whose last dimension runs over the partners and is
    summed), partner moments m[20]; the octupole difference m - ratio *
    octupole enters the correction (None: no correction)."""
    r2 = x[0] * x[0] + x[1] * x[1] + x[2] * x[2]
    ri = 1.0 / torch.sqrt(torch.clamp(r2, min=1.0e-20))
    d1, d2, d3 = ri ** 3, -3.0 * ri ** 5, 15.0 * ri ** 7

    def D2(a, b):
        return d2 * x[a] * x[b] + (d1 if a == b else 0.0)

    def D3(a, b, c):
        t = d3 * x[a] * x[b] * x[c]
        for u, v, w in ((a, b, c), (a, c, b), (b, c, a)):
            if u == v:
                t = t + d2 * x[w]
        return t

    D = [None] * 20
    D[0] = -ri
    for a in _R3:
        D[1 + a] = d1 * x[a]
        for b in range(a, 3):
            D[_I2[a][b]] = D2(a, b)
            for c in range(b, 3):
                D[_I3[a][b][c]] = D3(a, b, c)
    L = [m[0] * D[i] for i in range(rows)]
    for a in _R3:
        for b in _R3:
            L[0] = L[0] + 0.5 * m[_I2[a][b]] * D[_I2[a][b]]
            for c in _R3:
                L[0] = L[0] - m[_I3[a][b][c]] * D[_I3[a][b][c]] / 6.0
                L[1 + a] = L[1 + a] + 0.5 * m[_I2[b][c]] * D[_I3[a][b][c]]
        if dipole:   # DRHODT: the potential's dipole and the row sums of the second derivatives
            L[0] = L[0] - m[1 + a] * D[1 + a]
            L[1 + a] = L[1 + a] - m[1 + a] * (D[_I2[a][0]] + D[_I2[a][1]] + D[_I2[a][2]])
        for b in range(a, 3):
            if rows == 20:
                L[_I2[a][b]] = L[_I2[a][b]] - sum(m[1 + c] * D[_I3[a][b][c]] for c in _R3)
    C = None
    if ratio is not None:
        C = []
        for d in _R3:
            s = 0.0
            for a in _R3:
                for b in range(a, 3):
                    for c in range(b, 3):
                        mult = {1: 1.0, 2: 3.0, 3: 6.0}[len({a, b, c})] / 6.0
                        i = _I3[a][b][c]
                        w = mult * (m[i] - ratio * octupole[i - 10])
                        # the order-4 derivatives without their d4 term
                        u = 0.0
                        q = (a, b, c, d)
                        for p, r, e, f in ((0, 1, 2, 3), (0, 2, 1, 3), (0, 3, 1, 2), (1, 2, 0, 3), (1, 3, 0, 2),
                                           (2, 3, 0, 1)):
                            if q[p] == q[r]:
                                u = u + d3 * x[q[e]] * x[q[f]]
                                if q[e] == q[f] and p == 0:
                                    u = u + d2
                        s = s - w * u
            C.append(s.sum(-1))
    return [v.sum(-1) for v in L], C


def _order(a):
    """[n, 512, ...] -> [n, 64 coarse, 8 children, ...]"""
    n = a.shape[0]
    t = a.reshape((n, 4, 2, 4, 2, 4, 2) + a.shape[2:])
    t = t.permute((0, 1, 3, 5, 2, 4, 6) + tuple(range(7, t.dim())))
    return t.reshape((n, 64, 8) + a.shape[2:])


def _unorder(a):
    n = a.shape[0]
    t = a.reshape((n, 4, 4, 4, 2, 2, 2) + a.shape[3:])
    t = t.permute((0, 1, 4, 2, 5, 3, 6) + tuple(range(7, t.dim())))
    return t.reshape((n, CELLS) + a.shape[3:])


def _exact_level(nb, kind, tg, dx, theta, type_, M, com, mon, L, Lc):
    """Adds one level's interactions to L (and writes L_c) for the targets."""
    dev, rho = M.device, type_ == "rho"
    leaf = torch.as_tensor(kind == _abi.SLOT_LEAF, device=dev)
    src = M.clone()
    src[..., 0] += torch.where(leaf[:, None], mon, 0.0)
    src, cm, mo = _order(src), _order(com), _order(torch.where(leaf[:, None], mon, 0.0))
    nbt = torch.as_tensor(nb, device=dev).long()
    steps = [(d, f, n, *(torch.as_tensor(v, device=dev) for v in _coarse_step(d))) for d, f, n in _stencil(theta)]
    for is_leaf in (False, True):
        tall = torch.as_tensor(tg[(kind[tg] == _abi.SLOT_LEAF) == is_leaf], device=dev).long()
        for i in range(0, len(tall), 4096):
            t = tall[i:i + 4096]
            rows = 4 if is_leaf else 20
            outL = torch.zeros(len(t), 64, 8, rows, dtype=torch.float64, device=dev)
            outC = torch.zeros(len(t), 64, 8, 3, dtype=torch.float64, device=dev)
            for d, far, near, raw, cc in steps:
                s = nbt[t][:, raw]
                here = (s >= 0)[..., None]
                s = s.clamp(min=0)
                pl = leaf[s][..., None] & here
                m, y, p = src[s, cc], cm[s, cc], mo[s, cc]
                mt = m.movedim(-1, 0)
                yt = y.movedim(-1, 0)
                refined = (here & ~pl).any().item() if is_leaf else True
                for k in range(8):
                    f = torch.as_tensor(far[k], device=dev)
                    n = torch.as_tensor(near[k], device=dev)
                    if is_leaf:
                        on, any_ = here & ~pl & (f | n), refined
                        # p2p on the lattice
                        j = np.arange(8)
                        off = [2 * d[0] + ((j >> 2) & 1) - ((k >> 2) & 1), 2 * d[1] + ((j >> 1) & 1) - ((k >> 1) & 1),
                               2 * d[2] + (j & 1) - (k & 1)]
                        r = np.sqrt(np.maximum(sum(o * o for o in off), 1))
                        use = far[k] | near[k]
                        q = torch.where(pl, p, 0.0)
                        outL[:, :, k, 0] -= q @ torch.as_tensor(use / r / dx, device=dev)
                        for a in _R3:
                            outL[:, :, k, 1 + a] -= q @ torch.as_tensor(use * off[a] / r ** 3 / dx ** 2, device=dev)
                    else:
                        on, any_ = here & (f | (n & pl)), bool(far[k].any() or near[k].any())
                    if not any_:
                        continue
                    x = [torch.where(on, cm[t][:, :, k, a, None] - yt[a], 1.0) for a in _R3]
                    mm = [torch.where(on, v, 0.0) for v in mt]
                    ratio = oct_ = None
                    if rho:
                        ratio = 0.0 if is_leaf else mm[0] / src[t][:, :, k, 0, None]
                        oct_ = [0.0] * 10 if is_leaf else [src[t][:, :, k, 10 + c, None] for c in range(10)]
                    Ls, Cs = _pair_sums(x, mm, ratio, oct_, not rho, rows)
                    outL[:, :, k] += torch.stack(Ls, -1)
                    if rho:
                        outC[:, :, k] += torch.stack(Cs, -1)
            L[t, :, :rows] += _unorder(outL)
            if rho:
                has = (nbt[t] >= 0) & ~leaf[nbt[t].clamp(min=0)]
                has[:, 13] = not is_leaf
                write = t[has.any(1)] if is_leaf else t
                Lc[write] = _unorder(outC)[has.any(1)] if is_leaf else _unorder(outC)


def _exact_root(type_, theta, M, com, L, Lc):
    dev, rho = M.device, type_ == "rho"
    i = _unit_cells(dev)
    d2 = ((i[:, None] - i[None, :]) ** 2).sum(-1)
    on = (d2 > 0) & (1.0 / torch.sqrt(d2.clamp(min=1e-20)) <= theta)
    x = [torch.where(on, com[0, :, None, a] - com[0, None, :, a], 1.0) for a in _R3]
    mm = [torch.where(on, M[0, None, :, c], 0.0) for c in range(20)]
    ratio = mm[0] / M[0, :, 0, None] if rho else None
    Ls, Cs = _pair_sums(x, mm, ratio, [M[0, :, 10 + c, None] for c in range(10)], not rho, 20)
    L[0] += torch.stack(Ls, -1)
    if rho:
        Lc[0] = torch.stack(Cs, -1)


def _exact_m2m(lv, up, mon, xbase, M, com, pM, pcom, rho):
    """The upward pass of one level: leaf centres, then each coarse cell's
    moments about its centre of mass in the parent."""
    dev = M.device
    leaf = torch.as_tensor(lv.kind == _abi.SLOT_LEAF, device=dev)
    if rho:
        centre = xbase[:, None, :] + _unit_cells(dev) * lv.dx
        com[leaf] = centre[leaf]
    if up is None:
        return
    A = M.clone()
    A[..., 0] += torch.where(leaf[:, None], mon, 0.0)
    A, X = _order(A), _order(com)
    par, octant = torch.as_tensor(lv.parent, device=dev).long(), torch.as_tensor(lv.octant, device=dev).long()
    q = torch.arange(64, device=dev)
    cell = ((q // 16)[None] + 4 * (octant & 1)[:, None]) * 64 + ((q // 4 % 4)[None] + 4 * ((octant >> 1) & 1)[:, None]) * 8 \
        + (q % 4)[None] + 4 * ((octant >> 2) & 1)[:, None]
    if rho:
        Y = (A[..., :1] * X).sum(2) / A[..., :1].sum(2)
        pcom[par[:, None], cell] = Y
    else:
        Y = pcom[par[:, None], cell]
    r = X - Y[:, :, None, :]
    B = A.clone()
    for a in _R3:
        B[..., 1 + a] += A[..., 0] * r[..., a]
        for b in range(a, 3):
            B[..., _I2[a][b]] += A[..., 1 + a] * r[..., b] + A[..., 1 + b] * r[..., a] + A[..., 0] * r[..., a] * r[..., b]
            for c in range(b, 3):
                t = A[..., 0] * r[..., a] * r[..., b] * r[..., c]
                for u, v, w in ((a, b, c), (b, c, a), (c, a, b)):
                    t = t + A[..., _I2[u][v]] * r[..., w] + A[..., 1 + u] * r[..., v] * r[..., w]
                B[..., _I3[a][b][c]] += t
    pM[par[:, None], cell] = B.sum(2)


def _exact_l2l(lv, pL, pLc, pcom, com, L, Lc, rho):
    """Adds the parents' expansions, moved to the cells, to L and L_c."""
    dev = L.device
    par, octant = torch.as_tensor(lv.parent, device=dev).long(), torch.as_tensor(lv.octant, device=dev).long()
    i = torch.arange(CELLS, device=dev)
    cell = ((i // 128)[None] + 4 * (octant & 1)[:, None]) * 64 + ((i // 16 % 4)[None] + 4 * ((octant >> 1) & 1)[:, None]) * 8 \
        + (i // 2 % 4)[None] + 4 * ((octant >> 2) & 1)[:, None]
    A, r = pL[par[:, None], cell], com - pcom[par[:, None], cell]
    B = A.clone()
    for a in _R3:
        B[..., 0] += A[..., 1 + a] * r[..., a]
        for b in _R3:
            B[..., 0] += 0.5 * A[..., _I2[a][b]] * r[..., a] * r[..., b]
            B[..., 1 + a] += A[..., _I2[a][b]] * r[..., b]
            for c in _R3:
                t = A[..., _I3[a][b][c]]
                B[..., 0] += t * r[..., a] * r[..., b] * r[..., c] / 6.0
                B[..., 1 + a] += 0.5 * t * r[..., b] * r[..., c]
                if c >= a:
                    B[..., _I2[a][c]] += t * r[..., b]
    L += B
    if rho:
        Lc += pLc[par[:, None], cell]


def exact(case, seed):
    dev, rho = _device(), case["type"] == "rho"

    def zeros(n, *row):
        return torch.zeros((n, CELLS) + row, dtype=torch.float64, device=dev)

    if case["family"] == "dropin":
        lv = _dropin_level(case, seed)
        M, com, mon = (torch.as_tensor(a, device=dev) for a in (lv.M, lv.com, lv.mon))
        L, Lc = zeros(27, 20), zeros(27, 3)
        if case["entry"] == "root":
            _exact_root(case["type"], case["theta"], M[13:14], com[13:14], L[13:14], Lc[13:14])
        else:
            _exact_level(lv.neighbors, lv.kind, np.array([13]), lv.dx, case["theta"], case["type"], M, com, mon, L, Lc)
        return {"L": L[13].cpu().numpy(), "L_c": Lc[13].cpu().numpy()}
    if case["family"] == "level":
        nb, kind, xbase, dx, tg, c = _level_shape(case)
        M, com, mon = _level_state(case, seed)
        if case["partial"]:
            for s, cells in _halo_cells(case).items():
                gone = torch.ones(CELLS, dtype=torch.bool, device=dev)
                gone[torch.as_tensor(cells, device=dev).long()] = False
                for a in (M, mon) + ((com,) if kind[s] == _abi.SLOT_NONLEAF else ()):
                    a[s, gone] = 0.0
        L, Lc = zeros(len(kind), 20), zeros(len(kind), 3)
        _exact_level(nb, kind, tg, dx, case["theta"], case["type"], M, com, mon, L, Lc)
        return {"L": L, "L_c": Lc}

    levels = _tree_shape(case["shape"], case["max_level"], case["threshold"]).levels
    mass, rate = _tree_masses(case, seed)
    xb = [torch.as_tensor(lv.xbase, device=dev) for lv in levels]
    com = [zeros(lv.nnodes, 3) for lv in levels]
    for solve in ("rho",) if rho else ("rho", "drhodt"):
        src = mass if solve == "rho" else rate
        M = [zeros(lv.nnodes, 20) for lv in levels]
        for i in range(len(levels) - 1, -1, -1):
            up = levels[i - 1] if i else None
            _exact_m2m(levels[i], up, src[i], xb[i], M[i], com[i], M[i - 1] if i else None,
                       com[i - 1] if i else None, solve == "rho")
    out, L, Lc = [], [], []
    for i, lv in enumerate(levels):
        L.append(zeros(lv.nnodes, 20))
        Lc.append(zeros(lv.nnodes, 3))
        if i == 0 and lv.kind[0] == _abi.SLOT_NONLEAF:
            _exact_root(case["type"], 0.5, M[0], com[0], L[0], Lc[0])
        else:
            _exact_level(lv.neighbors, lv.kind, np.arange(lv.nnodes), lv.dx, 0.5, case["type"], M[i], com[i], src[i],
                         L[i], Lc[i])
        if i:
            _exact_l2l(lv, L[i - 1], Lc[i - 1], com[i - 1], com[i], L[i], Lc[i], rho)
        leaf = torch.as_tensor(lv.kind == _abi.SLOT_LEAF, device=dev)
        g = zeros(lv.nnodes, 4)
        g[..., 0] = torch.where(leaf[:, None], L[i][..., 0], 0.0)
        if rho:
            g[..., 1:] = torch.where(leaf[:, None, None], -(L[i][..., 1:4] + Lc[i]), 0.0)
        out.append({"M": M[i], "com": com[i], "L": L[i].clone(), "L_c": Lc[i], "g": g})
        if case["leaf_g_only"]:
            out[-1]["L"][leaf] = 0.0
        if not rho:
            out[-1] = {k: out[-1][k] for k in ("M", "L", "g")}
    return out
