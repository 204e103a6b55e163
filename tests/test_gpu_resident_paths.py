"""Which launches a solve takes: resident ones where the system fits the chip,
the launch per phase where it does not or where a resident launch had to leave.
The counts of the system's resident batches tell them apart, so that a solve
that quietly took the other way does not pass for one that was tested."""
import numpy as np
import pytest

import ogs5_amd as ox
from ogs5_amd import workloads as W

from test_gpu_resident import _scenario, _solve

pytestmark = pytest.mark.gpu


def test_one_workgroup_launches_keep_out_of_the_census_ring():
    """The census entries of a system's launches are used again after 64 of
    them, and cleared by the launches half a ring before.  A launch of one
    workgroup clears none, so it may not be numbered among them: here a launch
    that left (decision 2) is followed by 40 launches of one workgroup and then
    by more than a ring of counted ones, none of which may find its entry with
    the old decision and leave."""
    sc = _scenario("quad", (40, 40))  # CG: one workgroup; BiCGStab: several
    system = W.make_system(sc, ox.FP64)
    s = system[1]
    s.resident_leave(1)
    _solve(sc, system, False, method=ox.BICGSTAB)
    assert s.resident_counts()[1] == 1
    for _ in range(40):
        _solve(sc, system, False)
    run = s.resident_counts()[0]
    for _ in range(80):
        _solve(sc, system, False, method=ox.BICGSTAB)
    assert s.resident_counts() == (run + 80, 1)
    s.close()
