"""Buffers that share an allocation: replacing some of them gives their
memory back and leaves the others as they were, for handles whose buffers all
share one, that mix both kinds, and at the line between them (2 MiB: 3 doubles
per particle at 87,381 of them)."""
import numpy as np
import pytest

import _paths  # noqa: F401
from mfixdem import workloads
from mfixdem.system import DemSystem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 500, 12000, 87360, 87424])
def test_replaced_buffers_leave_the_rest(n):
    p, parts = workloads.lattice_member(n, 1.0e3, 0.9, 0.3, 3)

    def run(retune):
        s = DemSystem(p)
        s.set_particles(parts)
        s.init()
        s.run(1, 30)
        bytes_before = s.device_bytes()
        for _ in range(retune):
            s.set_tuning()
            assert s.device_bytes() == bytes_before
        s.run(31, 30)
        out = s.get_particles()
        s.close()
        return out

    for a, b in zip(run(0), run(3)):
        assert np.array_equal(a, b)
