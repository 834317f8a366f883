"""An inlet that runs out of slots in the very step in which an outlet deletes
particles.  The call reports MFIXDEM_ERR_CAPACITY as the oracle does, the
deletions of that step stand and free their slots, and the handle goes on:
step by step, within one call, and from new particles, bit for bit against
the oracle."""
import numpy as np
import pytest

import _paths  # noqa: F401
from mfixdem import abi, workloads
from mfixdem.system import DemSystem
from oracle_py import OracleSystem
from test_gpu_dem_bcs import D, RHO, assert_same, params
from test_gpu_parity import assert_same_pairs

pytestmark = pytest.mark.gpu

GONE = 240   # the step in which the layer below crosses the outlet
V = -0.5
CAPACITY = abi.ERRORS_BY_NAME["CAPACITY"]


def case(n, mi_start):
    """n spheres that leave in step GONE and no slot besides theirs; the inlet
    opens at mi_start."""
    box = (0.05, 0.016, 0.05)
    p = params(box, (10, 8, 10), grav=(0.0, 0.0, 0.0), max_pip=n)
    q = np.arange(n)
    pos = np.stack([0.003 + 0.0013 * (q % 33), np.full(n, 0.0012), 0.003 + 0.0013 * (q // 33)])
    parts = workloads.make_particles(pos, 0.5 * D, RHO,
                                     vel=np.tile([[0.0], [V], [0.0]], (1, n)))
    outlet = abi.dem_bc(abi.BC_MASS_OUTFLOW, abi.PLANE_N, (0.0, 0.0, 0.0), (box[0], 0.0, box[2]),
                        vel=[(0.0, V, 0.0)])
    inlet = abi.dem_bc(abi.BC_MASS_INFLOW, abi.PLANE_S, (0.02, box[1], 0.02),
                       (0.03, box[1], 0.03), vel=[(0.0, V, 0.0)], ep_s=[0.2])
    inlet.mi_start_time = mi_start
    return p, [outlet, inlet], parts


def begin(s, bcs, parts):
    s.set_particles(parts)
    s.set_dem_bcs(bcs, seed=11)
    s.init()


def code(call):
    with pytest.raises(abi.MfixDemError) as e:
        call()
    return e.value.code


@pytest.mark.parametrize("n", [1, 300, 900])
@pytest.mark.parametrize("one_call", [False, True])
def test_out_of_slots_in_a_step_that_deletes(n, one_call):
    dt = 1.0e-5
    p, bcs, parts = case(n, (GONE - 1.5) * dt)
    g, o = DemSystem(p), OracleSystem(p)
    for s in (g, o):
        begin(s, bcs, parts)
    if one_call:
        assert code(lambda: g.run(1, 2 * GONE)) == CAPACITY
        assert code(lambda: o.run(1, 2 * GONE)) == CAPACITY
    else:
        for s in (g, o):
            s.run(1, GONE - 1)
        assert_same(g, o, "before")
        assert code(lambda: g.step(GONE)) == CAPACITY
        assert code(lambda: o.step(GONE)) == CAPACITY
    # the outlet's deletions of that step stand; the oracle stops short of them
    pos, vel, om, st = g.get_particles()
    assert np.all(st == 0) and not pos.any() and not vel.any() and not om.any()
    assert np.all(o.get_particles()[3] == 3)
    # the freed slots are the inlet's: it seeds the lowest in the next step,
    # and what it seeds moves
    k = 40
    if n > 1:   # with one slot the next seed but one finds none again
        for nn in range(GONE + 1, GONE + 1 + k):
            g.step(nn)
            g.synchronize()
        pos, vel, om, st = g.get_particles()
        new = np.flatnonzero(st)
        assert new.size > 0 and np.array_equal(new, np.arange(new.size))
        assert np.all(vel[1, new] == V)
        y0 = pos[1, new].copy()
        g.run(GONE + 1 + k, k)
        y1 = g.get_particles()[0][1, new]
        assert np.allclose(y1 - y0, k * dt * V, rtol=1e-9, atol=0.0)
    # and from new particles
    o.close()
    p2, bcs2, parts2 = case(n, GONE * dt)
    o = OracleSystem(p2)
    for s in (g, o):
        begin(s, bcs2, parts2)
    nn = 1
    for steps in (GONE - 1, 1, 1, 59):
        for s in (g, o):
            try:
                s.run(nn, steps)
            except abi.MfixDemError as e:   # one slot: the second seed finds none
                assert n == 1 and e.code == CAPACITY
        nn += steps
        assert_same(g, o, f"after step {nn - 1}")
        if n == 1 and nn > GONE + 1:
            break
    if n > 1:
        assert_same_pairs(g, o)
    g.close()
    o.close()


@pytest.mark.parametrize("calls", [(300,), (239, 61), (240, 60), (1,) * 300])
def test_one_call_and_step_by_step_agree(calls):
    """Inside a call a step is queued ahead of the wait for the one before it,
    between calls none is: the same states and pairs however the steps are
    divided."""
    p, bcs, parts = case(300, 0.0)
    p.max_pip = 600
    g, o = DemSystem(p), OracleSystem(p)
    for s in (g, o):
        begin(s, bcs, parts)
    nn = 1
    for k in calls:
        g.run(nn, k)
        nn += k
    o.run(1, nn - 1)
    assert_same(g, o, f"{len(calls)} calls")
    assert_same_pairs(g, o)
    g.close()
    o.close()
