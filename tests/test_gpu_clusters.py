"""The two forms of the pair kernel (run on an MI355X): steps without
energies of small systems sum the pairs by clusters of eight, energy
evaluations with one wave to a chunk, in the same order and the same
arithmetic, so the forces of the two are equal to the bit."""
import copy
import ctypes as C

import numpy as np
import pytest

from blade_amd import system
from tests.helpers import spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("base,kw", [
    ("config1", {}),                                        # no lambda, box edge near twice the cutoff
    ("msld_small", {}),                                     # partly filled blocks, exclusions, lambda
    ("msld_small", {"soft_core": True}),
    ("msld_small", {"vdw_method": 1, "elec_method": 0}),
    ("msld_small", {"vdw_method": 2, "elec_method": 2}),
    ("config2_small", {}),
    ("config2_small", {"tile_chunk": 5}),                   # groups of eight tiles cut short
    ("two_site_small", {"soft_core": True, "tile_chunk": 16}),
] + [("msld_small", {"soft_core": True, "vdw_method": v, "elec_method": e}) for v in range(3) for e in range(3)])
def test_cluster_and_wave_forms_are_bit_identical(base, kw):
    sp = copy.copy(spec(base))
    for k, v in kw.items():
        setattr(sp, k, v)
    s = system.build(sp)
    s.run_energy()
    L, dev = s.L, s.device()

    def forces(energy):
        f = np.zeros(3 * sp.n + sp.nblocks, dtype=np.int64)
        assert L.bm_domdec_update(dev, 0) == 0
        assert L.bm_calc_force(dev, 0, energy) == 0
        assert L.bm_sync(dev) == 0
        assert L.bm_get_force_fixed(dev, f.ctypes.data_as(C.POINTER(C.c_longlong))) == 0
        return f

    wave, cluster = forces(1), forces(0)
    assert np.any(wave)
    assert np.array_equal(wave, cluster)
    s.close()
