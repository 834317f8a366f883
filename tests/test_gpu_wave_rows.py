"""The pair phase of the step kernel at its edges, bit for bit against the
oracle: wavefronts of 8, 16, 32 and 64 particles with a partly filled last
one, rows with no entry, contact queues that fill and wrap (dense beds), and
one row of more contacts than a batch of 64 holds.  Without gas both sides
do the same FP64 operations in the same order, so the tolerance is zero."""
import numpy as np
import pytest

import _paths  # noqa: F401
from mfixdem import abi, workloads
from mfixdem.system import DemSystem
from oracle_py import OracleSystem

pytestmark = pytest.mark.gpu


def dense(n, seed=3):
    """n nearly equal spheres on a body-centred lattice, neighbours overlapping."""
    rng = np.random.default_rng(seed)
    d = 1.0e-3 * rng.uniform(0.97, 1.0, n)
    a = 0.99e-3 * 2.0 / np.sqrt(3.0)
    m = max(1, int(np.ceil((n / 6.0) ** (1.0 / 3.0))))
    k = np.arange(n)
    q, c = k // 2, k % 2
    off = 0.25 + 0.5 * c
    pos = a * np.stack([q % m + off, q // (m * m) + off, (q // m) % m + off]) + 0.25e-3
    pos += 5.0e-6 * rng.uniform(-1.0, 1.0, (3, n))
    p, _, _ = workloads.settling_bed(n=1)
    p.max_pip = n
    p.xlength = p.zlength = m * a + 0.5e-3
    p.ylength = (q[-1] // (m * m) + 2) * a + 0.5e-3
    p.dtsolid = 2.0e-6
    perm = rng.permutation(n)
    return p, workloads.make_particles(pos[:, perm], 0.5 * d, 2500.0,
                                       vel=0.05 * rng.standard_normal((3, n)),
                                       omega=20.0 * rng.standard_normal((3, n)))


def big_sphere(n=150):
    """One sphere of 8 mm with n spheres of 1 mm pressed on it, in a spiral."""
    k = np.arange(n) + 0.5
    y = 1.0 - 2.0 * k / n
    t = np.pi * (1.0 + 5.0 ** 0.5) * k
    s = np.sqrt(1.0 - y * y)
    dirs = np.stack([s * np.cos(t), y, s * np.sin(t)])
    centre = np.array([[8.0e-3]] * 3)
    pos = np.concatenate([centre + 4.495e-3 * dirs, centre], axis=1)
    r = np.append(np.full(n, 0.5e-3), 4.0e-3)
    p, _, _ = workloads.settling_bed(n=1)
    p.max_pip = n + 1
    p.xlength = p.ylength = p.zlength = 16.0e-3
    p.max_radius = 4.0e-3
    p.dtsolid = 2.0e-6
    order = np.argsort(np.sin(37.0 * np.arange(n + 1)))   # the big one's id inside the range
    rng = np.random.default_rng(2)
    return p, workloads.make_particles(pos[:, order], r[order], 2500.0,
                                       vel=0.05 * rng.standard_normal((3, n + 1)),
                                       omega=20.0 * rng.standard_normal((3, n + 1)))


@pytest.mark.parametrize("n", [1, 7, 63, 65, 257, 4099, 30011, "big"])
def test_pair_phase_bit_exact(n):
    p, parts = big_sphere() if n == "big" else dense(n)
    g, o = DemSystem(p), OracleSystem(p)
    for s in (g, o):
        s.set_particles(parts)
        s.init()
        s.step(1)
    if n == "big":   # every small sphere starts in touch with the big one
        touching = np.count_nonzero(np.abs(o.get_pairs()[2]).sum(axis=1))
        assert touching > 128, touching
    for s in (g, o):
        s.run(2, 29)
    for a, b, what in zip(g.get_particles(), o.get_particles(), ("pos", "vel", "omega", "state")):
        assert np.array_equal(a, b), what
    gi, gn, gp = g.get_pairs()
    oi, on, op = o.get_pairs()
    assert np.array_equal(gi, oi) and np.array_equal(gn, on) and np.array_equal(gp, op)
    g.close()
    o.close()
