"""Lists longer than the tile kernels' window of 1,024 blocks (run on an
MI355X): rows whose tiles and exclusions lie in several windows, bit-exact
against the oracle's list, and the forces of both against each other with the
bar of the other parity tests (1e-5 relative RMS)."""
import ctypes as C

import numpy as np
import pytest

from blade_amd import synthetic, system
from oracle import oracle as orc
from tests.helpers import rel_rms

pytestmark = pytest.mark.gpu


def dilute(waters, spacing, seed):
    """water at low density: long lists whose forces the oracle sums quickly"""
    edge = spacing * int(np.ceil(round(waters ** (1 / 3), 9)))
    sp = synthetic.water_box(waters, (edge,) * 3, seed)[0]
    sp.rcut, sp.rswitch, sp.elec_method = 9.0, 8.0, 2
    return sp


def domdec(s):
    """slot order, blocks, tiles and masks of the device's list"""
    L, dev = s.L, s.device()
    nb, nt, ne = C.c_int(), C.c_int(), C.c_int()
    assert L.bm_get_domdec_sizes(dev, C.byref(nb), C.byref(nt), C.byref(ne)) == 0
    l2g, bc = np.zeros(32 * nb.value, np.int32), np.zeros(nb.value, np.int32)
    ti, tj, tm = np.zeros(nt.value, np.int32), np.zeros(nt.value, np.int32), np.zeros(32 * nt.value, np.uint32)
    i32, u32 = C.POINTER(C.c_int), C.POINTER(C.c_uint32)
    assert L.bm_get_domdec(dev, l2g.ctypes.data_as(i32), bc.ctypes.data_as(i32), ti.ctypes.data_as(i32),
                           tj.ctypes.data_as(i32), tm.ctypes.data_as(u32)) == 0
    return l2g, bc, np.stack([ti, tj], 1), tm.reshape(-1, 32)


# three windows and five
@pytest.mark.parametrize("waters,blocks", [(22000, 2049), (44000, 4097)])
def test_list_of_several_windows(waters, blocks):
    sp = dilute(waters, 6.5, 0xB1ADE0F8)
    s = system.build(sp)
    s.run_energy()
    top, rp = s.topology(), s.runparams()
    x = orc.rectify(top, rp, system.soa(sp.pos))
    want = orc.domdec(top, rp, x)
    got = domdec(s)
    ti, tj = want[3][:, 0], want[3][:, 1]
    far = (ti // 1024) != (tj // 1024)
    print("\n[%d atoms] blocks %d tiles %d, %d between windows, %d with exclusions" %
          (sp.n, len(want[2]), len(ti), far.sum(), np.any(want[4][far], axis=1).sum()), flush=True)
    assert len(want[2]) >= blocks and np.any(want[4][far])
    assert np.array_equal(s.positions(), want[0])
    for g, w in zip(got, want[1:]):
        assert np.array_equal(g, w)
    fo = orc.forces(top, rp, s.positions(), np.ones(1))[0]
    assert rel_rms(s.forces(), fo) <= 1e-5
    s.close()
