"""The two forms of the pair kernel (run on an MI355X): steps without
energies of small systems sum the pairs by clusters of eight, energy
evaluations with one wave to a chunk, in the same order and the same
arithmetic, so the forces of the two are equal to the bit."""
import copy
import ctypes as C

import numpy as np
import pytest

from blade_amd import system
from oracle import oracle as orc
from tests.helpers import rel_rms, spec

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


@pytest.mark.parametrize("soft", [False, True])
def test_lj_table_beyond_lds(soft):
    """more than 78 atom types (a table of more than 6,144 entries): both
    forms read it from global memory; against the oracle too (1e-5 relative
    RMS, 1e-6 of the pair energy)"""
    sp = copy.deepcopy(spec("msld_small"))
    sp.soft_core = soft
    oxygens = [i for i, a in enumerate(sp.atoms) if a[4] == "OT"][:90]
    for k, i in enumerate(oxygens):
        t = "O%02dX" % k
        a = list(sp.atoms[i])
        a[4] = t
        sp.atoms[i] = tuple(a)
        sp.types[t] = sp.types["OT"]
        sp.bond_par[("HT", t)] = next(v for key, v in sp.bond_par.items() if set(key) == {"OT", "HT"})
        sp.angle_par[("HT", t, "HT")] = sp.angle_par[("HT", "OT", "HT")]
        eps, rmin, eps14, rmin14, e14, comb = sp.nb_par["OT"]
        sp.nb_par[t] = (eps, rmin + 0.002 * k, eps14, rmin14, e14, comb)
    s = system.build(sp)
    s.run_energy()
    top, rp = s.topology(), s.runparams()
    assert top.contents.n_types ** 2 > 6144
    lam = orc.theta_to_lambda(top, rp, np.array(sp.theta0, float))
    fo, do, eo, pairs = orc.forces(top, rp, s.positions(), lam)
    fe, eg = s.forces(), s.energy()
    L, dev = s.L, s.device()
    f = np.zeros(3 * sp.n + sp.nblocks, dtype=np.int64)
    assert L.bm_domdec_update(dev, 0) == 0 and L.bm_calc_force(dev, 0, 0) == 0 and L.bm_sync(dev) == 0
    assert L.bm_get_force_fixed(dev, f.ctypes.data_as(C.POINTER(C.c_longlong))) == 0
    assert np.array_equal(fe, f[:3 * sp.n] / 2.0 ** 32)
    assert rel_rms(fe, fo) <= 1e-5
    assert abs(eg[7] - eo[7]) <= 1e-6 * abs(eo[7])
    s.close()
