"""Ensembles whose members' boxes are far larger than their spheres need:
their search cells grow instead of their number.  Each member evolves bit for
bit as in a handle of its own, which keeps the cells of the cut-off, and what
a box's cells cost in memory is bounded by the member's slots."""
import numpy as np
import pytest

import _paths  # noqa: F401
from mfixdem import abi, workloads
from mfixdem.ensemble import Ensemble
from mfixdem.system import DemSystem

pytestmark = pytest.mark.gpu


def member(n, box, cluster, seed):
    """n spheres spread over the box, or packed in one corner of it."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    q = np.arange(n)
    cell = np.stack([q % m, q // m % m, q // (m * m)])
    if cluster:
        pos = 0.6e-3 + 0.985e-3 * cell
    else:
        pos = (cell + 0.5) / m * np.array(box)[:, None]
        pos[:, 1::2] = pos[:, 0:2 * (n // 2):2] + np.array([[0.7e-3], [0.69e-3], [0.0]])
    p, _, _ = workloads.settling_bed(n=1)
    p.max_pip = n
    p.xlength, p.ylength, p.zlength = box
    p.desgridsearch_imax = p.desgridsearch_jmax = p.desgridsearch_kmax = 20
    p.neighbor_search_n = 10
    p.dtsolid = 2.0e-6
    perm = rng.permutation(n)
    return p, workloads.make_particles(pos[:, perm], 0.5e-3, 2500.0,
                                       vel=0.05 * rng.standard_normal((3, n)),
                                       omega=20.0 * rng.standard_normal((3, n)))


# cells per slot from below the bound (16) to far above it, one sphere, a
# member that fills its slots and one that does not
BOXES = [(1, (0.01, 0.01, 0.01)), (63, (0.02, 0.02, 0.02)), (64, (0.3, 0.01, 0.02)),
         (65, (0.1, 0.1, 0.1)), (300, (0.02, 0.02, 0.02)), (500, (0.24, 0.24, 0.24)),
         (700, (0.05, 0.4, 0.05))]


@pytest.mark.parametrize("cluster", [False, True])
@pytest.mark.parametrize("scale", [1.0, 1.7])
def test_members_as_in_their_own_handles(cluster, scale):
    made = [member(n, box, cluster, 3 + k) for k, (n, box) in enumerate(BOXES)]
    e = Ensemble([p for p, _ in made])
    for k, (_, parts) in enumerate(made):
        e.set_particles(k, parts)
    if scale != 1.0:
        e.set_tuning(cell_scale=scale)
    e.init()
    e.run(1, 35)
    contacts = 0
    for k, (p, parts) in enumerate(made):
        s = DemSystem(p)
        s.set_particles(parts)
        s.init()
        s.run(1, 5)   # (spheres that start overlapped are apart again in 20 steps)
        contacts += np.count_nonzero(np.abs(s.get_pairs()[2]).sum(axis=1))
        s.run(6, 30)
        for a, b, what in zip(e.get_particles(k), s.get_particles(),
                              ("pos", "vel", "omega", "state")):
            assert np.array_equal(a, b), (k, what)
        s.close()
    assert contacts > (500 if cluster else 50), contacts
    e.close()


def test_memory_follows_the_slots():
    """Four members of 500 spheres in 0.24 m: 8.1 million cells of the cut-off
    each, 8 bytes of cell range each if they were kept."""
    made = [member(500, (0.24, 0.24, 0.24), False, 3) for _ in range(4)]
    e = Ensemble([p for p, _ in made])
    assert e.device_bytes() < 4 * 8 * 8.1e6 / 4
    e.close()


def test_too_many_cells_stay_refused():
    """More than 1,022 cells of the cut-off along an axis."""
    p, _ = member(64, (1.3, 0.01, 0.01), False, 3)
    for make in (lambda: Ensemble([p, p]), lambda: DemSystem(p)):
        with pytest.raises(abi.MfixDemError) as err:
            make()
        assert err.value.code == abi.ERRORS_BY_NAME["UNSUPPORTED"]
