"""A server's memory budget counts what a request's solver allocates: the
FP64 iterates, the products in the build's precision (N gamma, r, J in both
orders, M^-1 D^T gamma and its exchanged copy, and in the mixed build D^T
gamma of four iterates and M^-1), the frames, and the partial sums per tile
in the form of the launches and of the resident passes."""
import pytest

from dvide_amd import scenes, system

pytestmark = pytest.mark.gpu

TILE_ROWS, TILE_BODIES, SLOTS, HEAVY = 512, 256, 8, 128


def solver_bytes(nc, nb, nbil, mixed):
    cap = max(1024, nc + nc // 4)  # of the scene's first collision detection
    rows, tiles = 3 * cap + nbil, -(-(cap + nbil) // TILE_ROWS)
    lipschitz = (-(-nb // TILE_BODIES) + 2 * cap // HEAVY + 2) // 2 * 2
    partials = 4 * SLOTS * tiles + 2 * SLOTS + 2 * lipschitz + (4 * SLOTS * tiles + 4 * lipschitz)
    products = 5 * rows + 8 + 4 * (2 * cap + nbil + 2 * nb) + 16
    if not mixed:
        return 8 * (partials + 5 * rows + 16 + products)
    products += 4 * 4 * nb + nb + 1
    return 8 * (partials + 5 * rows + 16) + 4 * products + 4 * 6 * cap


@pytest.mark.parametrize("build", [system.BUILD_FP64, system.BUILD_MIXED])
def test_two_requests_share_a_budget_that_holds_both(gpu, monkeypatch, build):
    monkeypatch.setenv("DVIDE_TUNE", "0")
    scs = [scenes.compaction(5, n=1200, width=1.2, lid=scenes.LID_BILATERAL), scenes.pile(31, 1500)]
    for short in (0, 1):
        members = [system.from_scene(sc, build, tol=1e-5, max_iterations=30) for sc in scs]
        need = 0
        for g, sc in zip(members, scs):
            g.step()
            st = g.stats()
            assert st.iterations > 0
            need += solver_bytes(st.num_contacts, len(sc.mass), len(sc.bil_dofs), build == system.BUILD_MIXED)
        srv = system.Server(build, max_slots=4, hbm_budget=float(need - short))
        for g in members:
            srv.submit(g)
        srv.poll()
        # admission clears a scene's statistics; a waiting one keeps its last step's
        assert members[0].stats().iterations == 0
        assert (members[1].stats().iterations > 0) == bool(short)
        assert len(srv.drain()) == 2
        srv.close()
        for g in members:
            g.close()
