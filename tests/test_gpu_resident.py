"""The resident passes against the passes as launches.

A slot whose team fits the chip keeps its contacts' state in registers for
thousands of passes; fixed rows per thread (DV_PARAM_ROWS_PER_THREAD) keep a
scene on the launches.  Both add in the same order, so every result is equal
bit for bit: around the edges of a row tile (512 rows), past one and two tiles
per CU (two rows per thread, and three), and with the rows and bodies that take paths of their
own (bilateral rows, a movable body with thousands of contacts, body units
without a movable body)."""
import copy

import numpy as np
import pytest

from dvide_amd import scenes, system

pytestmark = pytest.mark.gpu


def bits_equal(x, y):
    x = np.asarray(x, np.float64)
    y = np.asarray(y, np.float64)
    return x.shape == y.shape and np.array_equal(x.view(np.uint64), y.view(np.uint64))


def layer_of(n):
    """n spheres on a floor, one contact each."""
    sc = scenes.layer(7, per_side=int(np.ceil(np.sqrt(n))))
    for k in ("pos", "vel", "mass", "geom", "fixed", "family"):
        setattr(sc, k, getattr(sc, k)[:n + 1].copy())
    return sc


def landed_shell():
    sc = scenes.shell_bed(3, nx=8, ny=16, layers=1)
    sc.pos[:, 1] -= 1e-4
    return sc


def ball_on_a_layer():
    """A large sphere on some thirty small ones: more contacts than a round of
    a body's loads, fewer than make a body's sum a workgroup's."""
    sc = layer_of(256)
    sc.geom[-1, 0] = 2.0
    sc.pos[-1] = (0.0, 2.02, 0.0)
    return sc


SCENES = {
    "ball": scenes.ball_on_box,
    **{f"layer_{n}": (lambda n=n: layer_of(n)) for n in (63, 511, 512, 513, 1025)},
    "pile_6000": lambda: scenes.pile(31, 6000),
    "free_lid": lambda: scenes.compaction(5, n=3000, width=1.5, lid=scenes.LID_FREE),
    "bilateral_lid": lambda: scenes.compaction(5, n=1200, width=1.2, lid=scenes.LID_BILATERAL),
    "shell": landed_shell,
    "ball_on_a_layer": ball_on_a_layer,
    "box_58000": lambda: scenes.compaction(2002, n=58000, width=4.0, lid=scenes.LID_NONE),
    # past two rows per thread on 256 CUs
    "box_118000": lambda: scenes.compaction(2002, n=118000, width=5.1, lid=scenes.LID_NONE),
    "bilateral_118000": lambda: scenes.compaction(2002, n=118000, width=5.1, lid=scenes.LID_BILATERAL),
}


@pytest.mark.parametrize("build", [system.BUILD_FP64, system.BUILD_MIXED])
@pytest.mark.parametrize("name", SCENES)
def test_resident_passes_equal_the_launches(gpu, monkeypatch, name, build):
    monkeypatch.setenv("DVIDE_TUNE", "0")  # no solve is spent on measuring schedules
    sc = SCENES[name]()
    out = []
    for rows in (1, 0):
        g = system.from_scene(copy.deepcopy(sc), build, tol=1e-7, max_iterations=150)
        g.setRowsPerThread(rows)
        steps = []
        for _ in range(2):
            g.step()
            st = g.stats()
            steps.append((st.num_contacts, st.iterations, st.passes, st.backtracks, st.residual, st.objective))
        out.append((steps, g.gamma, g.v, g.p))
        g.close()
    assert out[0][0] == out[1][0]
    assert out[0][0][0][0] > 0
    for a, b in zip(out[0][1:], out[1][1:]):
        assert bits_equal(a, b)


def _launched(sc, build, steps):
    g = system.from_scene(copy.deepcopy(sc), build, tol=1e-7, max_iterations=150)
    g.setRowsPerThread(1)
    for _ in range(steps):
        g.step()
    out = (g.stats().iterations, g.gamma, g.v, g.p)
    g.close()
    return out


@pytest.mark.parametrize("how", ["batch", "server"])
@pytest.mark.parametrize("names", [("ball", "layer_513", "pile_6000", "bilateral_lid", "free_lid"),
                                   ("layer_63", "pile_6000", "box_58000", "shell", "box_58000", "layer_1025")])
def test_teams_side_by_side_equal_the_launches(gpu, monkeypatch, names, how):
    """Several scenes' teams in one launch (one row per thread, and with the
    large scenes, which outnumber the chip's CUs, two): every member as its
    launches alone leave it, whichever rows and neighbours it has."""
    monkeypatch.setenv("DVIDE_TUNE", "0")
    build, steps = system.BUILD_MIXED, 2
    scs = [SCENES[n]() for n in names]
    members = [system.from_scene(copy.deepcopy(sc), build, tol=1e-7, max_iterations=150) for sc in scs]
    if how == "batch":
        b = system.Batch(build)
        for g in members:
            b.add(g)
        for _ in range(steps):
            b.step()
        b.close()
    else:
        srv = system.Server(build, max_slots=4)
        for _ in range(steps):
            for g in members:
                srv.submit(g)
            assert len(srv.drain()) == len(members)
        srv.close()
    for sc, g in zip(scs, members):
        ref = _launched(sc, build, steps)
        assert g.stats().iterations == ref[0]
        for a, b in zip((g.gamma, g.v, g.p), ref[1:]):
            assert bits_equal(a, b)
        g.close()


@pytest.mark.parametrize("build", [system.BUILD_FP64, system.BUILD_MIXED])
@pytest.mark.parametrize("name", ["pile_6000", "bilateral_lid"])
def test_passes_past_one_launch_equal_the_launches(gpu, monkeypatch, name, build):
    """A launch runs 2048 passes; the next takes up the iterates, N gamma and
    M^-1 D^T gamma that it left in memory (also after a backtrack)."""
    monkeypatch.setenv("DVIDE_TUNE", "0")
    out = []
    for rows in (1, 0):
        g = system.from_scene(SCENES[name](), build, tol=1e-300, max_iterations=2500)
        g.setRowsPerThread(rows)
        g.step()
        st = g.stats()
        out.append(((st.iterations, st.passes, st.backtracks), g.gamma, g.v, g.p))
        g.close()
    assert out[0][0] == out[1][0]
    assert out[0][0][1] > 2048
    for a, b in zip(out[0][1:], out[1][1:]):
        assert bits_equal(a, b)
