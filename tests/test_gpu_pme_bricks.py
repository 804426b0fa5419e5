"""The PME spread's bricks (run on an MI355X): grids whose bricks take each
of the three side rules, whole axes, uneven bricks and overhangs on every
axis, against the FP64 oracle with the bars of the other parity tests
(forces <= 1e-5 relative RMS, energy <= 1e-6 relative)."""
import copy

import numpy as np
import pytest

from blade_amd import system
from oracle import oracle as orc
from tests.helpers import rel_rms, spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,grid", [
    (6, (18, 20, 24)),      # fewer than 64 bricks: the least side (5), uneven
    (8, (18, 18, 27)),      # least side 7, whose floor gives fewer bricks
    (4, (16, 27, 20)),      # least side 4 of order 4
    (6, (32, 36, 40)),      # side 8, uneven
    (4, (9, 64, 64)),       # an axis of few bricks beside long ones
    (6, (100, 90, 96)),     # more than 1,024 bricks of side 8: side 12
    (8, (90, 96, 100)),     # order 8 keeps side 8
])
def test_spread_bricks(order, grid):
    sp = copy.copy(spec("msld_small"))
    sp.order, sp.grid = order, grid
    s = system.build(sp)
    s.run_energy()
    top, rp = s.topology(), s.runparams()
    lam = orc.theta_to_lambda(top, rp, np.array(sp.theta0, float))
    fo, do, eo, pairs = orc.forces(top, rp, s.positions(), lam)
    fg, eg = s.forces(), s.energy()
    print("\n[order %d grid %s] force relRMS %.2e recip %.6f oracle %.6f" % (order, grid, rel_rms(fg, fo), eg[8], eo[8]),
          flush=True)
    assert rel_rms(fg, fo) <= 1e-5
    assert abs(eg[20] - eo[20]) <= 1e-6 * abs(eo[20])
    s.close()
