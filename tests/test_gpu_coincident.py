"""A solvent atom exactly on a soft-core substituent atom (run on an
MI355X): the pair's energy is finite and its force zero, and the other pairs
of the two atoms count as ever.  Forces, pair energy and dU/dlambda of both
forms of the pair kernel (energy and plain evaluations) against the FP64
oracle with the bars of the other parity tests; the pair energy differs from
that of a slightly displaced atom by far less than the bar."""
import copy
import ctypes as C

import numpy as np
import pytest

from blade_amd import system
from oracle import oracle as orc
from tests.helpers import coincident, rel_rms

pytestmark = pytest.mark.gpu

ENBDIRECT = 7


@pytest.mark.parametrize("vdw,elec", [(0, 1), (1, 0), (2, 2)])
def test_coincident_soft_core_atoms(vdw, elec):
    sp, a, o = coincident(vdw_method=vdw, elec_method=elec)
    s = system.build(sp)
    s.run_energy()
    top, rp = s.topology(), s.runparams()
    x = s.positions()
    assert all(x[k * sp.n + a] == x[k * sp.n + o] for k in range(3))
    lam = orc.theta_to_lambda(top, rp, np.array(sp.theta0, float))
    fo, do, eo, pairs = orc.forces(top, rp, x, lam)
    assert np.all(np.isfinite(fo)) and np.all(np.isfinite(eo))
    fe, eg, dg = s.forces(), s.energy(), s.dudl()
    L, dev = s.L, s.device()
    f = np.zeros(3 * sp.n + sp.nblocks, dtype=np.int64)
    assert L.bm_domdec_update(dev, 0) == 0 and L.bm_calc_force(dev, 0, 0) == 0 and L.bm_sync(dev) == 0
    assert L.bm_get_force_fixed(dev, f.ctypes.data_as(C.POINTER(C.c_longlong))) == 0
    print("\n[vdw %d elec %d] force relRMS %.2e pair energy %.6f oracle %.6f max |dU/dlambda diff| %.2e of %.1f"
          % (vdw, elec, rel_rms(fe, fo), eg[ENBDIRECT], eo[ENBDIRECT], np.max(np.abs(dg - do)), np.max(np.abs(do))),
          flush=True)
    assert np.array_equal(fe, f[:3 * sp.n] / 2.0 ** 32)
    assert rel_rms(fe, fo) <= 1e-5
    # the atoms' own forces too: they are not among the largest
    own = [k * sp.n + i for k in range(3) for i in (a, o)]
    assert rel_rms(fe[own], fo[own]) <= 1e-5
    assert abs(eg[ENBDIRECT] - eo[ENBDIRECT]) <= 1e-6 * abs(eo[ENBDIRECT])
    # soft-core dE/dr enters dU/dlambda in FP32
    assert np.max(np.abs(dg - do)) <= 1e-6 * np.max(np.abs(do))
    s.close()
