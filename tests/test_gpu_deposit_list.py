"""EP_G of the initial deposition (GARG_2012) against the oracle on both sides
of the size from which a thread takes two particles (131,072), with an odd
last one and a single particle.  The fixed-point sums hold EP_G to 1e-14, as
for the other depositions."""
import numpy as np
import pytest

import _paths  # noqa: F401
from mfixdem import abi
from mfixdem.system import DemSystem
from oracle_py import OracleSystem
from test_gpu_filter_tiles import case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cells", [(1, (4, 6, 4)), (25013, (16, 36, 16)),
                                     (131071, (28, 60, 28)), (131072, (28, 60, 28)),
                                     (131329, (28, 60, 28))])
def test_initial_fields(n, cells):
    p, parts, gas = case(n, cells, abi.INTERP_GARG_2012)
    d = abi.default_params()  # the options of the filter schemes back off
    p.des_interp_on, p.des_interp_mean_fields = d.des_interp_on, d.des_interp_mean_fields
    p.des_interp_width = d.des_interp_width
    g, o = DemSystem(p), OracleSystem(p)
    for s in (g, o):
        s.set_particles(parts)
        s.set_gas(gas)
        s.init()
    assert np.abs(g.get_gas()[0] - o.get_gas()[0]).max() <= 1e-14
    g.close()
    o.close()
