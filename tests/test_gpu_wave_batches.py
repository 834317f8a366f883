"""The pair phase of the step kernel in beds where every listed pair touches,
at 2, 4, 8, 16, 32 and 64 particles per wavefront (the last one partly
filled), bit for bit against the oracle: from 16 particles on a wavefront has
more contacts than a batch of 64 holds, so that rows are split across batches,
contacts are carried to the next one and the queue of 128 wraps, several
times over at 64.  Without gas both sides do the same FP64 operations in the
same order, so the tolerance is zero."""
import numpy as np
import pytest

import _paths  # noqa: F401
from mfixdem import workloads
from mfixdem.ensemble import Ensemble
from mfixdem.system import DemSystem
from oracle_py import OracleSystem

pytestmark = pytest.mark.gpu


def bed(n, seed=6):
    """n spheres on a body-centred lattice: 8 neighbours each that overlap, the
    next ones beyond the cut-off."""
    rng = np.random.default_rng(seed)
    d = 1.0e-3 * rng.uniform(0.98, 1.0, n)
    a = 0.965e-3 * 2.0 / np.sqrt(3.0)
    m = max(1, int(np.ceil((n / 2.0) ** (1.0 / 3.0))))
    k = np.arange(n)
    q, c = k // 2, k % 2
    off = 0.25 + 0.5 * c
    pos = a * np.stack([q % m + off, q // (m * m) + off, (q // m) % m + off]) + 0.25e-3
    pos += 3.0e-6 * rng.uniform(-1.0, 1.0, (3, n))
    p, _, _ = workloads.settling_bed(n=1)
    p.max_pip = n
    p.factor_rlm = 1.05
    p.xlength = p.zlength = m * a + 0.5e-3
    p.ylength = (q[-1] // (m * m) + 1) * a + 0.5e-3
    p.dtsolid = 1.0e-6
    p.neighbor_search_n = 6
    perm = rng.permutation(n)
    return p, workloads.make_particles(pos[:, perm], 0.5 * d, 2500.0,
                                       vel=0.02 * rng.standard_normal((3, n)),
                                       omega=20.0 * rng.standard_normal((3, n)))


def particles_per_wavefront(n, pairs):
    """The step kernel's choice for an uncoupled system."""
    room = max(2048.0, 1024.0 * (0.5 * pairs / n) ** 2)
    k = 6
    while k > 1 and n >> (k - 1) <= (room if k > 3 else 1024):
        k -= 1
    return 1 << k


def touching(o):
    return np.count_nonzero(np.abs(o.get_pairs()[2]).sum(axis=1))


@pytest.mark.parametrize("n, per", [(2011, 2), (4001, 4), (20021, 8), (50021, 16), (100003, 32),
                                    (140029, 64)])
def test_full_batches_bit_exact(n, per):
    p, parts = bed(n)
    g, o = DemSystem(p), OracleSystem(p)
    for s in (g, o):
        s.set_particles(parts)
        s.init()
        s.step(1)
    assert particles_per_wavefront(n, g.status().n_pairs) == per
    contacts = 2 * touching(o) / n * per   # both rows of a pair, in a wavefront
    if per >= 16:
        assert contacts > 100
    if per >= 32:
        assert contacts > 200
    for s in (g, o):
        s.run(2, 12)
    for a, b, what in zip(g.get_particles(), o.get_particles(), ("pos", "vel", "omega", "state")):
        assert np.array_equal(a, b), what
    gi, gn, gp = g.get_pairs()
    oi, on, op = o.get_pairs()
    assert np.array_equal(gi, oi) and np.array_equal(gn, on) and np.array_equal(gp, op)
    g.close()
    o.close()


def test_ensemble_of_full_batches_bit_exact():
    """The ensemble's kernel at 64 particles per wavefront: two members that
    end inside one, against the oracle."""
    made = [bed(n, seed) for n, seed in ((70001, 6), (70067, 7))]
    e = Ensemble([p for p, _ in made])
    for k, (_, parts) in enumerate(made):
        e.set_particles(k, parts)
    e.init()
    e.step(1)
    assert particles_per_wavefront(70016 + 70080, e.status().n_pairs) == 64
    e.run(2, 12)
    for k, (p, parts) in enumerate(made):
        o = OracleSystem(p)
        o.set_particles(parts)
        o.init()
        o.run(1, 13)
        for a, b, what in zip(e.get_particles(k), o.get_particles(),
                              ("pos", "vel", "omega", "state")):
            assert np.array_equal(a, b), (k, what)
        o.close()
    e.close()
