"""List columns past those that the scatter's workgroups scan for themselves
(run on an MI355X): a flat dilute box of more than 4,096 columns, alone and as
a batch member beside a box of few, bit-exact against the oracle's list and
its wrapped positions."""
import numpy as np
import pytest

from blade_amd import synthetic, system
from oracle import oracle as orc
from tests.helpers import rel_rms
from tests.test_gpu_list import domdec

pytestmark = pytest.mark.gpu


def flat(n, spacing, height, seed):
    """n x n waters in a flat box, one to a square of the given edge"""
    sp, rng = synthetic.water_box(n * n, (n * spacing, n * spacing, height), seed)
    pos = np.array(sp.pos).reshape(-1, 3, 3)
    at = rng.permutation(n * n)
    o = np.stack([at // n + 0.5, at % n + 0.5, np.zeros(n * n)], 1) * spacing
    o[:, 2] = rng.uniform(0.0, height, n * n)
    sp.pos = (pos - pos[:, :1] + o[:, None]).reshape(-1, 3)
    sp.rcut, sp.rswitch, sp.elec_method = 9.0, 8.0, 2
    sp.vel = synthetic._maxwell(rng, [a[6] for a in sp.atoms], sp.temperature)
    return sp


def columns(sp):
    a = (32 * np.prod(sp.box) / sp.n) ** (1 / 3)
    return int(np.ceil(sp.box[0] / a)) * int(np.ceil(sp.box[1] / a))


# many rounds of the scan, and either side of the line
@pytest.mark.parametrize("n,least,most", [(78, 900, 1024), (162, 4000, 4096), (166, 4097, 5000)])
def test_list_of_many_columns(n, least, most):
    sp = flat(n, 7.0, 11.0, 0xB1ADE0F9)
    assert least <= columns(sp) <= most
    s = system.build(sp)
    s.run_energy()
    top, rp = s.topology(), s.runparams()
    want = orc.domdec(top, rp, orc.rectify(top, rp, system.soa(sp.pos)))
    assert np.array_equal(s.positions(), want[0])
    for g, w in zip(domdec(s), want[1:]):
        assert np.array_equal(g, w)
    assert rel_rms(s.forces(), orc.forces(top, rp, s.positions(), np.ones(1))[0]) <= 1e-5
    s.close()


def test_batch_of_few_and_many_columns():
    """a batch's rebuild (step 10) against those of its members run alone, to
    the bit"""
    specs = [flat(20, 7.0, 11.0, 5), flat(166, 7.0, 11.0, 6), flat(24, 7.0, 11.0, 7)]
    assert [columns(sp) > 4096 for sp in specs] == [False, True, False]
    alone, members = [[system.build(sp) for sp in specs] for _ in range(2)]
    for s in alone + members:
        s.run_energy()   # device system and first list
    for s in alone:
        assert s.L.bm_dynamics(s.device(), 1, 12, 0, 1) == 0
    b = system.Batch(members)
    b.dynamics(1, 12)
    b.sync()
    for s, m in zip(alone, members):
        assert np.array_equal(s.positions(), m.positions())
        for g, w in zip(domdec(m), domdec(s)):
            assert np.array_equal(g, w)
    b.close()
    for s in alone + members:
        s.close()
