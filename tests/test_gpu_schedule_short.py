"""The schedule tuner after solves too short to measure: a class's eighth ends
the measuring for solves that run resident (which need no schedule), and a
later long solve that runs as launches still measures, decides and writes its
schedule."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_CHILD = r"""
import json, os, sys
sys.path.insert(0, %(root)r)
from dvide_amd import scenes, system
g = system.from_scene(scenes.pile(33, 8000), system.BUILD_MIXED, tol=1e-6, max_iterations=3)
p, v, steps = g.p, g.v, []
def step():  # from the same state, so that the rows stay in one class
    g.set_vector(system.VEC_P, p)
    g.set_vector(system.VEC_V, v)
    g.step()
    steps.append([g.stats().schedule_tuning, int(g.residentPasses > 0)])
for _ in range(10):
    step()
g.solver.maxIterations = 20000
os.environ["DVIDE_TEAM_WAIT_MS"] = "0"  # the next solve's team gives up, and those after it do not try
for _ in range(4):
    step()
print("RESULT " + json.dumps(steps))
"""


def test_short_solves_do_not_end_the_measuring_of_launches(gpu, tmp_path):
    path = tmp_path / "schedules.txt"
    env = dict(os.environ, DVIDE_SCHEDULE_FILE=str(path))
    env.pop("DVIDE_TUNE", None)
    r = subprocess.run([sys.executable, "-c", _CHILD % {"root": ROOT}], capture_output=True, text=True, timeout=100, env=env)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    steps = json.loads([x for x in r.stdout.splitlines() if x.startswith("RESULT ")][-1][7:])
    assert steps[:8] == [[1, 0]] * 8  # measured, as launches
    assert steps[8:10] == [[0, 1]] * 2  # resident
    assert steps[10] == [0, 0] and steps[11] == [1, 0]  # the team gave up; the next solve measures
    assert steps[13] == [0, 0]  # the class is decided
    assert len(path.read_text().split()) >= 6  # key rpt xcd wgc wgb score
