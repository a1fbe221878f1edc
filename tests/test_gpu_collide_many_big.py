"""More big geometries than one grid of their chunks holds: 140,000 boxes and
64 spheres, each resting on one box.  The (box, chunk of partners) pairs are
9.6 million workgroups, more than one launch takes; the contacts are known by
construction."""
import numpy as np
import pytest

from dvide_amd import scenes, system

pytestmark = pytest.mark.gpu


def test_boxes_past_one_grid(gpu):
    boxes, spheres, r, half, sink = 140000, 64, 0.05, 0.2, 1e-3
    n = boxes + spheres
    rng = np.random.default_rng(29)
    order = rng.permutation(n)  # body order: boxes and spheres mixed
    k = np.arange(boxes)
    side = int(np.ceil(np.sqrt(boxes)))
    pos = np.zeros((n, 3))
    pos[:boxes] = np.stack([k % side, np.zeros(boxes), k // side], 1)
    under = rng.choice(boxes, spheres, replace=False)
    pos[boxes:] = pos[under] + (0.0, half + r - sink, 0.0)
    geom = np.zeros((n, 3))
    geom[:boxes], geom[boxes:, 0] = half, r
    mass = rng.uniform(0.5, 2.0, n)
    fixed = np.r_[np.ones(boxes), np.zeros(spheres)].astype(np.int32)
    place = np.empty(n, int)  # of each geometry in the body order
    place[order] = np.arange(n)
    sc = scenes.cloud(1, n=8)
    sc.pos, sc.vel, sc.geom, sc.mass, sc.fixed = pos[order], np.zeros((n, 3)), geom[order], mass[order], fixed[order]
    sc.family = np.full(n, -1, np.int32)
    sc.bil_dofs, sc.bil_info = np.zeros((0, 2), np.int32), np.zeros((0, 2))
    g = system.from_scene(sc, system.BUILD_FP64, geom_mode=0)
    assert g.assemble() == spheres
    a, b, nap, _ = g.contacts()
    pairs = np.sort(np.stack([place[boxes:], place[under]], 1), axis=1)
    by = np.lexsort((pairs[:, 1], pairs[:, 0]))
    assert np.array_equal(np.stack([a, b], 1).astype(int), pairs[by])
    assert np.abs(nap[:, 3] + sink).max() < 1e-12
    # one contact to a sphere, its box fixed: N is the spheres' 1 / m
    x = rng.normal(size=3 * spheres)
    y = g.schur_product(x)
    assert np.abs(y - x / np.repeat(mass[boxes:][by], 3)).max() < 1e-12
    g.close()
