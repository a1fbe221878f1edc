"""Memory that calls borrow: the vectors of Schur products and the pinned
memory of set_vector and vector.  It does not grow with the scenes that have
called, and calls of several threads on scenes of different sizes get blocks
of their own."""
import ctypes
import threading

import numpy as np
import pytest

from dvide_amd import scenes, system

pytestmark = pytest.mark.gpu


def free_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_products_of_many_scenes_share_their_vectors(gpu):
    sc = scenes.pile(31, 12000)
    systems = [system.from_scene(sc, system.BUILD_FP64) for _ in range(40)]
    for g in systems:
        g.assemble()
    x = np.random.default_rng(3).normal(size=systems[0].vector(system.VEC_R).size)
    ref = systems[0].schur_product(x)
    for g in systems:  # whatever a scene's first launches of these kernels take
        assert np.array_equal(g.schur_product_noalloc(x), ref)
    before = free_bytes()
    for g in systems:  # each would hold 16 bytes a row of its own: 0.5 MB and more
        assert np.array_equal(g.schur_product(x), ref)
    assert before - free_bytes() <= 4 << 20
    for g in systems:
        g.close()


def test_threads_borrow_blocks_of_their_own(gpu):
    sizes = (300, 900, 2500, 7000, 15000, 300, 25000, 2500)
    systems = [system.from_scene(scenes.pile(50 + i, n), system.BUILD_FP64) for i, n in enumerate(sizes)]
    want = []
    for i, g in enumerate(systems):
        g.assemble()
        rng = np.random.default_rng(i)
        x, v = rng.normal(size=g.vector(system.VEC_R).size), rng.normal(size=g.v.size)
        want.append((x, v, g.schur_product(x)))
    wrong = []

    def work(i):
        g, (x, v, y) = systems[i], want[i]
        for k in range(20):
            g.set_vector(system.VEC_V, v * k)
            if not (np.array_equal(g.schur_product(x), y) and np.array_equal(g.v, v * k)):
                wrong.append((i, k))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(systems))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    for g in systems:
        g.close()


def test_product_without_rows_is_zero(gpu):
    """A scene whose contacts have gone keeps r's length; no row writes the
    product, which must not be what the vectors' memory held before."""
    other = system.from_scene(scenes.pile(31, 900), system.BUILD_FP64)
    other.assemble()
    g = system.from_scene(scenes.ball_on_box(), system.BUILD_FP64)
    g.step()
    n = g.vector(system.VEC_R).size
    assert n == 3
    p = g.p
    p[1::3][np.asarray(g.fixed()) == 0] += 10.0
    g.set_vector(system.VEC_P, p)
    assert g.assemble() == 0
    for product in (g.schur_product, g.schur_product_noalloc):
        other_product = other.schur_product if product == g.schur_product else other.schur_product_noalloc
        assert np.abs(other_product(np.ones(other.vector(system.VEC_R).size))).max() > 0
        assert np.array_equal(product(np.ones(n)), np.zeros(n))
    other.close()
    g.close()
