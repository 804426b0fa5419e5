"""Pair energies at the ends of the erfc table (run on an MI355X): arguments
past 6, a single row, and soft-core distances beyond a short cutoff, against
the FP64 oracle (the bar of the other parity tests, 1e-6 relative)."""
import copy

import numpy as np
import pytest

from blade_amd import system
from oracle import oracle as orc
from tests.helpers import spec

pytestmark = pytest.mark.gpu

ENBDIRECT = 7


@pytest.mark.parametrize("beta,rcut,rswitch", [
    (0.34, 9.0, 8.0),     # 49 rows of LDS
    (0.80, 9.0, 8.0),     # arguments to 7.2
    (1.50, 9.5, 8.0),     # to 14.25, where the energies vanish
    (0.30, 3.5, 3.0),     # a cutoff shorter than the soft radius
    (0.005, 9.0, 8.0),    # one row
])
def test_pair_energies_at_the_ends_of_the_erfc_table(beta, rcut, rswitch):
    sp = copy.copy(spec("msld_small"))
    sp.beta, sp.rcut, sp.rswitch, sp.soft_core = beta, rcut, rswitch, True
    s = system.build(sp)
    s.run_energy()
    top, rp = s.topology(), s.runparams()
    lam = orc.theta_to_lambda(top, rp, np.array(sp.theta0, float))
    eo = orc.forces(top, rp, s.positions(), lam)[2]
    eg = s.energy()
    print("\n[beta %g rcut %g] pair energy %.9f oracle %.9f" % (beta, rcut, eg[ENBDIRECT], eo[ENBDIRECT]), flush=True)
    assert abs(eg[ENBDIRECT] - eo[ENBDIRECT]) <= 1e-6 * abs(eo[ENBDIRECT])
    s.close()
