"""Results brought to the host: particles in global-id order with any
leading dimension, any subset of the arrays, at sizes around the chunks the
copies go through (512 KiB, four in flight), for one system and for the
members of an ensemble.  Right after mfixdem_init nothing has moved, so the
arrays equal the inputs bit for bit."""
import numpy as np
import pytest

import _paths  # noqa: F401
from mfixdem import abi, workloads
from mfixdem.ensemble import Ensemble
from mfixdem.system import DemSystem

pytestmark = pytest.mark.gpu


def bed(n, seed=1):
    p, parts = workloads.lattice_member(n, 1.0e3, 0.9, 0.3, seed)
    rng = np.random.default_rng(seed)
    perm = rng.permutation(n)
    return p, workloads.make_particles(parts.pos[:, perm], parts.radius, parts.ro_sol,
                                       vel=rng.standard_normal((3, n)),
                                       omega=rng.standard_normal((3, n)))


@pytest.mark.parametrize("n", [1, 7181, 7183, 28728, 60001])
def test_particles_come_back_at_any_size(n):
    p, parts = bed(n)
    s = DemSystem(p)
    s.set_particles(parts)
    s.init()
    want = (parts.pos, parts.vel, parts.omega)
    for got, a in zip(s.get_particles(), want):
        assert np.array_equal(got, a)
    ld = n + 13
    out = [np.full((3, ld), -7.0) for _ in range(3)]
    st = np.full(ld, -7, dtype=np.int8)
    for keep in ((0, 1, 2), (1,), (0, 2), ()):
        for a in out:
            a[:] = -7.0
        st[:] = -7
        ptr = [abi.dptr(out[k] if k in keep else None) for k in range(3)]
        abi.check(s.lib.mfixdem_get_particles(s.h, *ptr, abi.bptr(st if 1 not in keep else None),
                                              ld), "get_particles")
        for k in range(3):
            assert np.array_equal(out[k][:, :n], want[k]) if k in keep else (out[k] == -7.0).all()
            assert (out[k][:, n:] == -7.0).all()
        assert (st[:n] == (1 if 1 not in keep else -7)).all() and (st[n:] == -7).all()
    s.close()


def test_ensemble_members_come_back():
    members = [bed(n, seed) for n, seed in ((5003, 2), (17, 3), (9001, 4))]
    e = Ensemble([p for p, _ in members])
    for k, (_, parts) in enumerate(members):
        e.set_particles(k, parts)
    e.init()
    for k in (2, 0, 1):
        got = e.get_particles(k)
        for a, b in zip(got, (members[k][1].pos, members[k][1].vel, members[k][1].omega)):
            assert np.array_equal(a, b)
        assert (got[3] == 1).all()
    e.close()


def test_a_readback_between_binning_and_neighbour_search_changes_nothing():
    p, parts = bed(3001)
    pairs = []
    for read in (False, True):
        s = DemSystem(p)
        s.set_particles(parts)
        s.init()
        s.desgrid_pic()
        if read:
            s.get_particles()
        s.neighbour()
        pairs.append(s.get_pairs())
        s.close()
    for a, b in zip(*pairs):
        assert np.array_equal(a, b)
