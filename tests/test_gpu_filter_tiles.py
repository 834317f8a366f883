"""The filter schemes' deposition and gas-side drag against the oracle where
the LDS tile of a workgroup covers its cells (a packed bed), where it does
not (a few particles all over a large grid), and with one particle.
Tolerances as for the schemes elsewhere: EP_G 1e-14 (fixed-point sums), the
drag sums, added with atomics on both sides, 1e-12 of the largest value."""
import numpy as np
import pytest

import _paths  # noqa: F401
from mfixdem import abi, workloads
from mfixdem.system import DemSystem
from oracle_py import OracleSystem

pytestmark = pytest.mark.gpu


def case(n, cells, scheme):
    rng = np.random.default_rng(n)
    box = [2.0e-3 * c for c in cells]
    m = int(np.ceil((n / np.prod(cells)) ** (1.0 / 3.0) * max(cells))) + 1
    grid = [max(1, int(c * m / max(cells)) + 1) for c in cells]
    k = rng.permutation(int(np.prod(grid)))[:n]
    idx = np.stack([k % grid[0], (k // grid[0]) % grid[1], k // (grid[0] * grid[1])])
    step = np.array([b / g for b, g in zip(box, grid)])
    assert n <= np.prod(grid) and step.min() > 1.0e-3
    pos = (idx + 0.5) * step[:, None] + 0.4 * (step.min() - 1.0e-3) * rng.uniform(-1, 1, (3, n))
    p, _, _ = workloads.fluidised_bed(n=1, cells=cells, lx=box[0], ly=box[1], lz=box[2],
                                      dg=(0, 0, 0))
    p.max_pip = n
    p.max_radius = 0.5e-3
    p.interp_scheme = scheme
    p.des_interp_on = p.des_interp_mean_fields = 1
    if scheme != abi.INTERP_LINEAR_HAT:
        p.des_interp_width = 2.0e-3
    parts = workloads.make_particles(pos, 0.5e-3, 2500.0, vel=0.1 * rng.standard_normal((3, n)))
    return p, parts, workloads.frozen_gas(p)


@pytest.mark.parametrize("scheme", [abi.INTERP_LINEAR_HAT, abi.INTERP_SQUARE_DPVM],
                         ids=["hat", "dpvm"])
@pytest.mark.parametrize("n,cells", [(1, (4, 6, 4)), (300, (24, 48, 24)), (2500, (8, 20, 8))])
def test_deposition_and_drag(n, cells, scheme):
    p, parts, gas = case(n, cells, scheme)
    g, o = DemSystem(p), OracleSystem(p)
    for s in (g, o):
        s.set_particles(parts)
        s.set_gas(gas)
        s.init()
    assert np.abs(g.get_gas()[0] - o.get_gas()[0]).max() <= 1e-14
    for a, b in zip(g.drag_gs_gas(), o.drag_gs_gas()):
        assert np.abs(a - b).max() <= 1e-12 * max(np.abs(b).max(), 1e-300)
    g.run(1, 3)
    o.run(1, 3)
    for a, b in zip(g.get_particles()[:2], o.get_particles()[:2]):
        assert np.abs(a - b).max() <= 1e-12
    g.close()
    o.close()
