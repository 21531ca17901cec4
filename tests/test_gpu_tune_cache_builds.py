"""The file OCTOFMM_TUNE_CACHE names, read by a later process: a choice under this
build's key is taken as it stands, one under a key of other kernels (an earlier
library's, without the id of its sources) is not: the plan is tuned afresh and its
choice appended.

A process reads the file once, so each step is a process of its own.
"""
import os
import re
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
from octotiger_amd import _abi, hip, native, workloads
ctx = native.Context(theta=0.5, device=0)
lv = workloads.uniform_level((5, 4, 3), ((1, 4), (1, 3), (1, 2)), 20261801)
dl = hip.LevelOnDevice(lv)
plan = dl.plan(ctx, type_=_abi.RHO, flags=_abi.PLAN_AUTOTUNE)
print("variant", plan.stats()["variant"], flush=True)
plan.close()
dl.free()
ctx.close()
"""


def plan_with(path):
    """(variant of an autotuned plan, the file's lines) with the cache at path."""
    env = dict(os.environ, OCTOFMM_TUNE_CACHE=str(path))
    env.pop("OCTOFMM_VARIANT", None)
    r = subprocess.run([sys.executable, "-c", CHILD], cwd=ROOT, env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    return int(re.search(r"variant (\d+)", r.stdout).group(1)), path.read_text().split("\n")[:-1]


def test_choices_of_other_kernels_are_passed_over(tmp_path):
    path = tmp_path / "tune.txt"
    picked, lines = plan_with(path)
    key, variant = lines[0].split()
    assert len(lines) == 1 and int(variant) == picked
    path.write_text(f"{key} 2\n")
    assert plan_with(path) == (2, [f"{key} 2"])
    old = re.sub(r"/k[^/]*$", "", key)
    path.write_text(f"{old} 2\n")
    picked, lines = plan_with(path)
    assert len(lines) == 2 and lines[1].split() == [key, str(picked)]
