"""Which solves run resident, and teams of the sizes between a few workgroups
and half the chip.

A comparison of resident passes with passes as launches says nothing where
both sides are launches, so every case here states how many rows per thread
its team has (0: none, the scene runs as launches) and the passes that ran
resident are counted.  The sizes are those at which the kernel takes another
branch: a team of more than 64 members (FP64 forms a unit's sums ahead of the
decision up to there), members with several body tiles (a shell's contact
points), one, two and three rows per thread, and FP64 past its last."""
import copy

import numpy as np
import pytest

from dvide_amd import scenes, system
from tests.helpers import tiny_scene

pytestmark = pytest.mark.gpu

FP64, MIXED = system.BUILD_FP64, system.BUILD_MIXED


def bits_equal(x, y):
    x = np.asarray(x, np.float64)
    y = np.asarray(y, np.float64)
    return x.shape == y.shape and np.array_equal(x.view(np.uint64), y.view(np.uint64))


def box(n):
    return scenes.compaction(2002, n=n, width=5.0 * (n / 112000.0) ** (1.0 / 3.0), lid=scenes.LID_NONE)


def wide_shell():
    """640 spheres landed on a shell of 480 elements: few contacts, 70 body tiles."""
    sc = scenes.shell_bed(3, nx=16, ny=30, per_side=(16, 40), layers=1)
    sc.pos[:, 1] -= 1e-4
    return sc


def layer(n):
    """n spheres on a floor, one contact each."""
    sc = scenes.layer(7, per_side=int(np.ceil(np.sqrt(n))))
    for k in ("pos", "vel", "mass", "geom", "fixed", "family"):
        setattr(sc, k, getattr(sc, k)[:n + 1].copy())
    return sc


def among(sc, n):
    """The scene and n free spheres far above it that touch nothing."""
    k, r = np.arange(n), 0.05
    side = int(np.ceil(np.sqrt(n)))
    pos = np.stack([3 * r * (k % side), np.full(n, 50.0), 3 * r * (k // side)], 1)
    for name, more in (("pos", pos), ("vel", np.zeros((n, 3))), ("mass", np.ones(n)), ("geom", np.tile([[r, 0.0, 0.0]], (n, 1))),
                       ("fixed", np.zeros(n, np.int32)), ("family", np.full(n, -1, np.int32))):
        setattr(sc, name, np.concatenate([getattr(sc, name), more]).astype(more.dtype))
    return sc


SCENES = {
    "ball": scenes.ball_on_box,
    # bodies decide the team's size: 16 members of which one has rows, and 256
    # of which 134 have two tiles each
    "few_contacts": lambda: among(layer(100), 7900),
    "many_bodies": lambda: among(box(58000), 150000),
    "pile_6000": lambda: scenes.pile(31, 6000),
    "wide_shell": wide_shell,
    "box_8000": lambda: box(8000),     # 36 members
    "box_17000": lambda: box(17000),   # 77
    "box_58000": lambda: box(58000),   # two rows a thread on 256 CUs
    "box_118000": lambda: box(118000),  # mixed three, FP64 none
    "bilateral_lid": lambda: scenes.compaction(5, n=1200, width=1.2, lid=scenes.LID_BILATERAL),
}


def _stepped(sc, build, rows, steps=2):
    g = system.from_scene(copy.deepcopy(sc), build, tol=1e-7, max_iterations=150)
    g.setRowsPerThread(rows)
    out = []
    for _ in range(steps):
        g.step()
        st = g.stats()
        out.append((st.num_contacts, st.iterations, st.passes, st.backtracks, st.residual, st.objective))
    ran = (g.residentPasses, g.teamRows, g.stats().passes)
    vectors = (g.gamma, g.v, g.p)
    g.close()
    return out, vectors, ran


@pytest.mark.parametrize("name,build,rows", [
    ("ball", FP64, 1), ("wide_shell", FP64, 1), ("wide_shell", MIXED, 1),
    ("box_8000", FP64, 1), ("box_8000", MIXED, 1), ("box_17000", FP64, 1), ("box_17000", MIXED, 1),
    ("few_contacts", FP64, 1), ("few_contacts", MIXED, 1), ("many_bodies", FP64, 2), ("many_bodies", MIXED, 2),
    ("box_58000", FP64, 2), ("box_58000", MIXED, 2), ("box_118000", FP64, 0), ("box_118000", MIXED, 3)])
def test_team_sizes_equal_the_launches(gpu, monkeypatch, name, build, rows):
    monkeypatch.setenv("DVIDE_TUNE", "0")
    sc = SCENES[name]()
    launched, ref, ran = _stepped(sc, build, 1)
    assert ran[0] == 0 and ran[1] == 0 and ran[2] > 0  # fixed rows per thread: as launches
    assert launched[0][0] > 0
    stats, vectors, ran = _stepped(sc, build, 0)
    assert ran == ((ran[2], rows, ran[2]) if rows else (0, 0, ran[2]))
    assert stats == launched
    for a, b in zip(ref, vectors):
        assert bits_equal(a, b)


@pytest.mark.parametrize("how", ["batch", "server"])
@pytest.mark.parametrize("build", [FP64, MIXED])
def test_scenes_side_by_side_run_resident(gpu, monkeypatch, build, how):
    """One row per thread beside each other, and with a scene past the chip's
    CUs two for all."""
    monkeypatch.setenv("DVIDE_TUNE", "0")
    for names, rows in ((("ball", "pile_6000", "bilateral_lid", "wide_shell", "few_contacts"), 1), (("pile_6000", "box_58000", "ball"), 2)):
        scs = [SCENES[n]() for n in names]
        members = [system.from_scene(copy.deepcopy(sc), build, tol=1e-7, max_iterations=150) for sc in scs]
        if how == "batch":
            b = system.Batch(build)
            for g in members:
                b.add(g)
            b.step()
            b.close()
        else:
            srv = system.Server(build, max_slots=4)
            for g in members:
                srv.submit(g)
            assert len(srv.drain()) == len(members)
            srv.close()
        for n, sc, g in zip(names, scs, members):
            launched, ref, _ = _stepped(sc, build, 1, steps=1)
            st = g.stats()
            assert g.residentPasses == st.passes > 0, n
            # (a server's slots end at different times, and a team is formed for those left)
            assert g.teamRows == rows if how == "batch" else g.teamRows in (1, rows), n
            assert (st.num_contacts, st.iterations, st.passes) == launched[0][:3], n
            for x, y in zip((g.gamma, g.v, g.p), ref):
                assert bits_equal(x, y), n
            g.close()


def test_passes_counts_are_read_only(gpu):
    g = system.from_scene(SCENES["ball"](), FP64)
    assert g.residentPasses == 0 and g.teamRows == 0
    for p in (system.PARAM_RESIDENT_PASSES, system.PARAM_TEAM_ROWS):
        with pytest.raises(system.DvideError) as e:
            g._set(p, 1)
        assert e.value.code == system.DV_ERR_ARG
    g.close()


@pytest.mark.parametrize("build", [FP64, MIXED])
def test_few_contacts_among_many_bodies_take_no_longer(gpu, monkeypatch, build):
    """100 contacts among 8,000 movable bodies: a pass on the one member that
    the rows need took 2.0 (FP64) and 2.6 times as long as one as launches,
    and on the sixteen that the bodies get takes 0.8 and 0.7 times as long."""
    monkeypatch.setenv("DVIDE_TUNE", "0")
    us = []
    for rows in (1, 0):
        g = system.from_scene(SCENES["few_contacts"](), build, tol=1e-300, max_iterations=200)
        g.setRowsPerThread(rows)
        best = np.inf
        for _ in range(6):
            g.step()
            best = min(best, 1e3 * g.stats().ms_solve / g.stats().passes)
        us.append(best)
        g.close()
    assert us[1] < 1.3 * us[0], us


def star(n):
    """A sphere whose x is tied to those of n others: n bilateral rows of one body."""
    pos = np.stack([0.3 * np.arange(n + 1), np.full(n + 1, 5.0), np.zeros(n + 1)], 1)
    return tiny_scene(pos, [[0.05, 0, 0]] * (n + 1), bilaterals=[(0, 3 * i, 0.0, 0.0) for i in range(1, n + 1)])


@pytest.mark.parametrize("build", [FP64, MIXED])
@pytest.mark.parametrize("n,alone,beside", [(12, 1, 1), (13, 0, 1), (32, 0, 1), (33, 0, 0)])
def test_bodies_with_many_bilateral_rows_run_as_launches(gpu, monkeypatch, build, n, alone, beside):
    """A body's bilateral rows are awaited in turn: past 12 a scene alone, past
    32 scenes beside each other take longer resident (with 49 rows 30 us a pass
    against 16 as launches)."""
    monkeypatch.setenv("DVIDE_TUNE", "0")
    launched, ref, _ = _stepped(star(n), build, 1)
    stats, vectors, ran = _stepped(star(n), build, 0)
    assert (ran[0] > 0) == bool(alone) and stats == launched
    for a, b in zip(ref, vectors):
        assert bits_equal(a, b)
    members = [system.from_scene(sc, build, tol=1e-7, max_iterations=150) for sc in (star(n), SCENES["ball"]())]
    b = system.Batch(build)
    for g in members:
        b.add(g)
    for _ in range(2):
        b.step()
    b.close()
    assert (members[0].residentPasses > 0) == bool(beside)
    for x, y in zip((members[0].gamma, members[0].v, members[0].p), ref):
        assert bits_equal(x, y)
    for g in members:
        g.close()


@pytest.mark.parametrize("build", [FP64, MIXED])
def test_a_team_that_cannot_be_placed_runs_as_launches(gpu, monkeypatch, build):
    """With no time to wait for its members a team of several workgroups gives
    up (every kernel exits at once): the step's passes run as launches, the
    next 16 solves do not try, and then the team forms."""
    monkeypatch.setenv("DVIDE_TUNE", "0")
    sc = layer(1025)
    ref = system.from_scene(copy.deepcopy(sc), build, tol=1e-7, max_iterations=40)
    ref.setRowsPerThread(1)
    g = system.from_scene(copy.deepcopy(sc), build, tol=1e-7, max_iterations=40)
    ran = []
    for k in range(18):
        if k == 0:
            monkeypatch.setenv("DVIDE_TEAM_WAIT_MS", "0")
        else:
            monkeypatch.delenv("DVIDE_TEAM_WAIT_MS", raising=False)
        ref.step()
        g.step()
        assert (g.stats().iterations, g.stats().residual) == (ref.stats().iterations, ref.stats().residual)
        for a, b in zip((g.gamma, g.v, g.p), (ref.gamma, ref.v, ref.p)):
            assert bits_equal(a, b)
        ran.append(g.residentPasses)
    assert ran[:17] == [0] * 17 and ran[17] == g.stats().passes > 0
    ref.close()
    g.close()


@pytest.mark.parametrize("build", [FP64, MIXED])
def test_a_batch_whose_teams_cannot_be_placed_runs_as_launches(gpu, monkeypatch, build):
    """A team of one workgroup needs no wait and runs on, those of several
    give up; every scene's result is that of its launches."""
    monkeypatch.setenv("DVIDE_TUNE", "0")
    monkeypatch.setenv("DVIDE_TEAM_WAIT_MS", "0")
    names = ("pile_6000", "ball", "bilateral_lid")
    members = [system.from_scene(SCENES[n](), build, tol=1e-7, max_iterations=150) for n in names]
    b = system.Batch(build)
    for g in members:
        b.add(g)
    b.step()
    b.close()
    for n, g in zip(names, members):
        launched, ref, _ = _stepped(SCENES[n](), build, 1, steps=1)
        st = g.stats()
        assert (st.num_contacts, st.iterations, st.passes) == launched[0][:3], n
        assert g.residentPasses == (st.passes if n == "ball" else 0), n
        for x, y in zip((g.gamma, g.v, g.p), ref):
            assert bits_equal(x, y), n
        g.close()


@pytest.mark.parametrize("build", [FP64, MIXED])
def test_a_server_whose_teams_cannot_be_placed_runs_as_launches(gpu, monkeypatch, build):
    """Freshly admitted slots whose teams give up, alone and beside a slot
    whose team (one workgroup) forms in every turn: the next turns run as
    launches.  The turns are bounded, so that a server that tries the teams
    for ever fails here."""
    monkeypatch.setenv("DVIDE_TUNE", "0")
    monkeypatch.setenv("DVIDE_TEAM_WAIT_MS", "0")
    for names in (("pile_6000", "bilateral_lid"), ("ball", "pile_6000")):
        members = [system.from_scene(SCENES[n](), build, tol=1e-7, max_iterations=150) for n in names]
        if names[0] == "ball":  # this one iterates for long
            members[0].solver.tolerance, members[0].solver.maxIterations = 1e-300, 20000
        srv = system.Server(build, max_slots=2)
        for g in members:
            srv.submit(g)
        done, turns = [], 0
        while srv.pending() and turns < 2000:
            done += srv.poll()
            turns += 1
            if len(done) == 1 and names[0] == "ball":  # the pile, beside the ball
                assert members[1].stats().iterations > 0 and members[0].stats().iterations == 0
        assert sorted(done) == [1, 2]
        srv.close()
        for n, g in zip(names, members):
            if n == "ball":
                continue
            launched, ref, _ = _stepped(SCENES[n](), build, 1, steps=1)
            st = g.stats()
            assert (st.num_contacts, st.iterations, st.passes) == launched[0][:3], n
            assert g.residentPasses == 0, n
            for x, y in zip((g.gamma, g.v, g.p), ref):
                assert bits_equal(x, y), n
        for g in members:
            g.close()


@pytest.mark.parametrize("build", [FP64, MIXED])
@pytest.mark.parametrize("name", ["pile_400", "bilateral_box"])
def test_a_solve_that_changes_between_resident_and_launches(gpu, monkeypatch, name, build):
    """A scene of one workgroup in a server starts resident, goes on as
    launches while another scene's team gives up beside it, and ends resident:
    the bits of its launches alone."""
    monkeypatch.setenv("DVIDE_TUNE", "0")
    sc = scenes.pile(33, 400) if name == "pile_400" else scenes.compaction(5, n=150, width=0.6, lid=scenes.LID_BILATERAL)

    def made():
        return system.from_scene(copy.deepcopy(sc), build, tol=1e-300, max_iterations=3000)

    ref = made()
    ref.setRowsPerThread(1)
    ref.step()
    assert 0 < ref.stats().num_contacts <= 512 - 3
    g, other = made(), system.from_scene(SCENES["pile_6000"](), build, tol=1e-300, max_iterations=100)
    monkeypatch.setenv("DVIDE_TEAM_WAIT_MS", "0")
    srv = system.Server(build, max_slots=2)
    srv.submit(g)
    for _ in range(4):
        srv.poll()
    srv.submit(other)
    assert len(srv.drain()) == 2
    srv.close()
    st = g.stats()
    assert (st.iterations, st.passes, st.backtracks, st.residual) == (
        ref.stats().iterations, ref.stats().passes, ref.stats().backtracks, ref.stats().residual)
    assert 0 < g.residentPasses < st.passes and other.residentPasses == 0
    for a, b in zip((g.gamma, g.v, g.p), (ref.gamma, ref.v, ref.p)):
        assert bits_equal(a, b)
    for s in (ref, g, other):
        s.close()
