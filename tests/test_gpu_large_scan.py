"""The scans behind a rebuild at sizes whose tile totals are summed in groups
(more than 4,096 tiles of 1,024 elements) and just below: search cells of a
dilute box, and slots of a system with a large capacity.  Touching pairs are
spread over the whole box, in its first and last cells among them, so that a
wrong offset loses or invents pairs.  Bit for bit against the oracle."""
import numpy as np
import pytest

import _paths  # noqa: F401
from mfixdem import abi, workloads
from mfixdem.system import DemSystem
from oracle_py import OracleSystem
from test_gpu_parity import assert_same_pairs

pytestmark = pytest.mark.gpu

# search cell of 1 mm spheres
CUT = abi.default_params().factor_rlm * 1.0e-3 * (1.0 + 1.0e-9)


def spread(cells, n_pairs=600, seed=4):
    """Touching pairs in a box of the given number of search cells per axis."""
    box = [(c - 2.5) * CUT for c in cells]
    rng = np.random.default_rng(seed)
    k = np.arange(n_pairs)
    m = int(np.ceil(n_pairs ** (1.0 / 3.0)))
    slot = np.stack([k % m, k // m % m, k // (m * m)]) / (m - 1)
    lo, hi = np.full(3, 1.5e-3), np.array(box) - 1.5e-3
    mid = lo[:, None] + slot * (hi - lo)[:, None]
    axis = rng.standard_normal((3, n_pairs))
    axis *= 0.495e-3 / np.sqrt((axis * axis).sum(axis=0))
    pos = np.concatenate([mid + axis, mid - axis], axis=1)
    n = 2 * n_pairs
    perm = rng.permutation(n)
    p, _, _ = workloads.settling_bed(n=1)
    p.max_pip = n
    p.xlength, p.ylength, p.zlength = box
    p.desgridsearch_imax = p.desgridsearch_jmax = p.desgridsearch_kmax = 20
    p.neighbor_search_n = 10
    p.dtsolid = 2.0e-6
    parts = workloads.make_particles(pos[:, perm], 0.5e-3, 2500.0,
                                     vel=0.05 * rng.standard_normal((3, n)),
                                     omega=20.0 * rng.standard_normal((3, n)))
    return p, parts


def compare(p, parts, capacity):
    o = OracleSystem(p)
    p.max_pip = capacity
    g = DemSystem(p)
    for s in (g, o):
        s.set_particles(parts)
        s.init()
    for s in (g, o):
        s.run(1, 25)
    for a, b, what in zip(g.get_particles(), o.get_particles(), ("pos", "vel", "omega", "state")):
        assert np.array_equal(a[..., :parts.n], b), what
        assert not np.any(a[..., parts.n:]), what
    assert g.status().rebuilds == o.status().rebuilds
    return g, o


# tiles of the cells and one more: 4,081; 4,097 with one element in the last,
# which is a group by itself; 5,121
@pytest.mark.parametrize("cells", [(128, 128, 255), (128, 128, 256), (320, 128, 128)])
def test_many_search_cells(cells):
    p, parts = spread(cells)
    g, o = compare(p, parts, parts.n)
    oi, on, _ = o.get_pairs()
    assert on.size >= parts.n // 2
    assert_same_pairs(g, o)
    g.close()
    o.close()


# tiles of the slots: 4,096 (summed directly), 4,097, 5,121
@pytest.mark.parametrize("capacity", [4096 * 1024, 4096 * 1024 + 1, 5120 * 1024 + 1])
def test_many_slots(capacity):
    p, parts = spread((40, 60, 50), n_pairs=4000)
    g, o = compare(p, parts, capacity)
    assert g.status().n_pairs == o.status().n_pairs >= parts.n // 2
    g.close()
    o.close()
