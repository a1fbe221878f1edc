"""Rows and threads of the resident passes whose inputs are not there: a scene
whose only rows are bilateral has no contact frames, so what their memory
holds (here those of a contact without a normal, from an earlier step) must
not reach the threads without a contact."""
import numpy as np
import pytest

from dvide_amd import system
from tests.helpers import tiny_scene

pytestmark = pytest.mark.gpu


def _after_a_contact_without_a_normal(build, rows_per_thread):
    # a sphere whose centre lies inside a fixed box: the contact's frame is NaN
    sc = tiny_scene([[0.0, 0.0, 0.0], [0.0, 0.1, 0.0]], [[1.0, 0.2, 1.0], [0.1, 0.0, 0.0]], fixed=[1, 0],
                    bilaterals=[(3, -1, 0.3, 0.0), (5, -1, -0.2, 0.0)])
    g = system.from_scene(sc, build, tol=1e-10, max_iterations=200)
    g.setRowsPerThread(rows_per_thread)
    with pytest.raises(system.DvideError) as e:
        g.step()
    assert e.value.code == -6  # DV_ERR_DIVERGED
    p = g.p
    p[4] = 3.0  # clear of the box
    g.set_vector(system.VEC_P, p)
    g.set_vector(system.VEC_V, np.zeros(6))
    g.set_vector(system.VEC_GAMMA, np.zeros(g.gamma.size))
    out = []
    for _ in range(2):
        g.step()
        st = g.stats()
        assert st.num_contacts == 0 and np.isfinite(st.residual)
        out.append((st.iterations, st.residual, g.gamma, g.v, g.p))
    g.close()
    return out


@pytest.mark.parametrize("build", [system.BUILD_FP64, system.BUILD_MIXED])
def test_only_bilateral_rows_after_a_contact_without_a_normal(gpu, build):
    resident, launches = (_after_a_contact_without_a_normal(build, r) for r in (0, 1))
    for a, b in zip(resident, launches):
        assert a[:2] == b[:2]
        for x, y in zip(a[2:], b[2:]):
            assert np.array_equal(x, y)
