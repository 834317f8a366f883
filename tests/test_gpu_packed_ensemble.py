"""Ensembles of thousands of systems smaller than a wavefront, whose slots
follow each other (from 1,536 systems on, while they fill half of their
wavefronts at most) and on the other side of that line: members of different
parameters, sizes and free slots side by side in one wavefront, each bit for
bit as alone, in either precision; a sphere outside the box is removed from
its own member only."""
import numpy as np
import pytest

import _paths  # noqa: F401
from mfixdem import abi, workloads
from mfixdem.ensemble import Ensemble
from mfixdem.system import DemSystem
from oracle_py import OracleSystem

pytestmark = pytest.mark.gpu


def member(cap, n, k, precision=abi.FP64, rogue=False):
    """n overlapping spheres in a box of their own, capacity cap; parameters
    by k."""
    rng = np.random.default_rng(100 + k)
    m = max(1, int(np.ceil(n ** (1.0 / 3.0))))
    q = np.arange(n)
    pos = 0.6e-3 + 0.985e-3 * np.stack([q % m, q // m % m, q // (m * m)]).astype(float)
    pos += 5.0e-6 * rng.uniform(-1.0, 1.0, (3, n))
    if rogue:
        pos[:, -1] = (-1.0e-3, 0.6e-3, 0.6e-3)
    p, _, _ = workloads.settling_bed(n=1)
    p.max_pip = cap
    p.precision = precision
    p.remove_rogue = 1
    p.xlength, p.zlength = m * 1.0e-3 + 0.5e-3, (m + k % 3) * 1.0e-3 + 0.5e-3
    p.ylength = (1 + k % 2) * m * 1.0e-3 + 0.5e-3
    p.neighbor_search_n = 10
    p.kn = p.kn_w = 700.0 + 100.0 * k
    p.mew = p.mew_w = 0.1 + 0.05 * k
    p.des_en_input[0] = p.des_en_wall_input[0] = 0.8 + 0.02 * k
    p.grav[:] = [0.3 * k, -9.81, -0.2 * k]
    p.dtsolid = 2.0e-6 + 1.0e-7 * k
    return p, workloads.make_particles(pos, 0.5e-3, 2000.0 + 100.0 * k,
                                       vel=0.05 * rng.standard_normal((3, n)),
                                       omega=20.0 * rng.standard_normal((3, n)))


def alone(kind, p, parts):
    s = kind(p)
    s.set_particles(parts)
    s.init()
    s.run(1, 45)
    out = s.get_particles()
    rebuilt = s.status()
    s.close()
    return out, rebuilt


def check(variants, count, kind):
    """An ensemble of count members that repeat the variants."""
    e = Ensemble([variants[k % len(variants)][0] for k in range(count)])
    for k in range(count):
        e.set_particles(k, variants[k % len(variants)][1])
    e.init()
    e.run(1, 45)
    want = [alone(kind, *v) for v in variants]
    for k in range(count):
        for a, b, what in zip(e.get_particles(k), want[k % len(variants)][0],
                              ("pos", "vel", "omega", "state")):
            assert np.array_equal(a, b), (k, what)
    per = np.bincount(np.arange(count) % len(variants), minlength=len(variants))
    assert e.status().rogue_deleted == sum(
        int(c) * w[1].rogue_deleted for c, w in zip(per, want))
    return e, want


# capacities, members, whether their slots follow each other
LINES = [((32,) * 8, 1536, True), ((32,) * 8, 1535, False), ((32,) * 7 + (33,), 1536, False),
         ((1, 64), 1600, False), ((1, 63), 1600, True), ((1,), 3001, True)]


@pytest.mark.parametrize("caps, count, packed", LINES)
def test_both_sides_of_the_line(caps, count, packed):
    variants = [member(c, c, k) for k, c in enumerate(caps)]
    e, _ = check(variants, count, OracleSystem)
    slots = sum(caps[k % len(caps)] for k in range(count))
    if caps[0] == 32:   # what a slot takes, empty ones counted with the others
        assert (e.device_bytes() < 2600 * slots) == packed
    e.close()


@pytest.mark.parametrize("precision", [abi.FP64, abi.MIXED])
def test_members_of_all_sizes_share_wavefronts(precision):
    caps = [(1, 1), (3, 2), (20, 20), (65, 65), (2, 1), (40, 33), (7, 7), (130, 90), (5, 5),
            (1, 1), (4, 3), (12, 12)]
    variants = [member(c, n, k, precision, rogue=k in (2, 5)) for k, (c, n) in enumerate(caps)]
    kind = OracleSystem if precision == abi.FP64 else DemSystem
    e, want = check(variants, 1709, kind)
    assert [w[1].rogue_deleted for w in want] == [int(k in (2, 5)) for k in range(len(caps))]
    e.close()


@pytest.mark.parametrize("tuning", [(1.0, abi.ROWS_WAVE128), (1.6, abi.ROWS_WAVE192),
                                    (2.5, abi.ROWS_THREAD)])
def test_tuning_choices_of_a_packed_ensemble(tuning):
    variants = [member(c, c, k) for k, c in enumerate((1, 20, 3, 40, 7, 30))]
    e = Ensemble([variants[k % 6][0] for k in range(1800)])
    for k in range(1800):
        e.set_particles(k, variants[k % 6][1])
    e.set_tuning(*tuning)
    e.init()
    e.run(1, 25)
    want = []
    for p, parts in variants:
        o = OracleSystem(p)
        o.set_particles(parts)
        o.init()
        o.run(1, 25)
        want.append(o.get_particles())
        o.close()
    for k in list(range(0, 1800, 7)) + [1799]:
        for a, b, what in zip(e.get_particles(k), want[k % 6], ("pos", "vel", "omega", "state")):
            assert np.array_equal(a, b), (k, what)
    e.close()
