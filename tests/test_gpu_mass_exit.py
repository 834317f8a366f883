"""Many particles leaving through an outlet in one step, around the 256 whose
ids reach the host with the count, while an inlet fills the freed slots:
bit for bit against the oracle."""
import numpy as np
import pytest

import _paths  # noqa: F401
from mfixdem import abi, workloads
from test_gpu_dem_bcs import D, RHO, assert_same, params, start
from test_gpu_parity import assert_same_pairs

pytestmark = pytest.mark.gpu


def layer(n):
    box = (0.05, 0.016, 0.05)
    p = params(box, (10, 8, 10), grav=(0.0, 0.0, 0.0), max_pip=n + 400)
    q = np.arange(n)
    pos = np.stack([0.003 + 0.0013 * (q % 33), np.full(n, 0.0012), 0.003 + 0.0013 * (q // 33)])
    vel = np.tile([[0.0], [-0.5], [0.0]], (1, n))
    parts = workloads.make_particles(pos, 0.5 * D, RHO, vel=vel)
    outlet = abi.dem_bc(abi.BC_MASS_OUTFLOW, abi.PLANE_N, (0.0, 0.0, 0.0), (box[0], 0.0, box[2]),
                        vel=[(0.0, -0.5, 0.0)])
    inlet = abi.dem_bc(abi.BC_MASS_INFLOW, abi.PLANE_S, (0.02, box[1], 0.02),
                       (0.03, box[1], 0.03), vel=[(0.0, -0.5, 0.0)], ep_s=[0.2])
    return start(p, [outlet, inlet], parts)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 900])
def test_layer_leaves_at_once(n):
    g, o = layer(n)
    nn = 1
    for k in (200, 39, 1, 1, 1, 58, 100):
        g.run(nn, k)
        o.run(nn, k)
        nn += k
        assert_same(g, o, f"after step {nn - 1}")
        # the layer is there before step 240 and gone after it
        assert (o.get_particles()[3] == 3).sum() == (n if nn <= 240 else 0)
    assert_same_pairs(g, o)
    g.close()
    o.close()


@pytest.mark.parametrize("last", [239, 240, 241, 400])
@pytest.mark.parametrize("n", [1, 257, 900])
def test_layer_leaves_within_one_call(n, last):
    """The deletions (step 240) overtake a step that is already queued, unless
    the call ends there."""
    g, o = layer(n)
    for s in (g, o):
        s.run(1, last)
    assert_same(g, o, f"after step {last}")
    for s in (g, o):
        s.run(last + 1, 60)
    assert_same(g, o, f"after step {last + 60}")
    assert_same_pairs(g, o)
    g.close()
    o.close()
