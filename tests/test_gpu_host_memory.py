"""Host memory of destroyed systems (run on an MI355X): the pinned staging of
a system's host transfers (8 bytes per degree of freedom) is given back, so
the process does not grow with the systems it has created and destroyed."""
import ctypes as C

import numpy as np
import pytest

from blade_amd import system
from tests.helpers import spec

pytestmark = pytest.mark.gpu


def _vmsize():
    with open("/proc/self/status") as f:
        return next(1024 * int(line.split()[1]) for line in f if line.startswith("VmSize"))


def test_destroyed_systems_leave_no_pinned_memory():
    sp = spec("config2")
    s = system.build(sp)
    s.prepare()
    top, rp = s.topology(), s.runparams()
    x, theta = system.soa(sp.pos), np.zeros(sp.nblocks)
    ptr = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))

    def systems(n):
        for _ in range(n):
            dev = C.c_void_p()
            assert s.L.bm_system_create(0, top, rp, ptr(x), None, ptr(theta), None, C.byref(dev)) == 0
            assert s.L.bm_system_destroy(dev) == 0

    systems(10)   # the runtime's own pools
    before = _vmsize()
    systems(20)
    grown = _vmsize() - before
    print("\n20 systems: %d bytes" % grown, flush=True)
    # their staging is 20 x 565 KB
    assert grown < 20 * 8 * 3 * sp.n / 4
    s.close()
