"""The branches of a step's graph (run on an MI355X): PME transforms in line,
on a branch of their own (6,000 atoms and more, 9,000 on the MFMA form) and ahead of a pair kernel
that takes the branch (grids without a square y-z plane), on either side of
the size line.  Forces and energy of the state after 30 replayed steps
against the FP64 oracle with the bars of the other parity tests (forces
<= 1e-5 relative RMS, energy <= 1e-6 relative), and the steps launched one
by one to the bit."""
import copy
import functools

import numpy as np
import pytest

from blade_amd import synthetic, system
from oracle import oracle as orc
from tests.helpers import rel_rms, relaxed

pytestmark = pytest.mark.gpu


@functools.lru_cache(maxsize=None)
def _water(nwat):
    box = (3 * nwat / synthetic.WATER_DENSITY) ** (1 / 3)
    sp, rng = synthetic.water_box(nwat, (box, box, box), 0xB1ADE0F0)
    sp.order, sp.temperature = 6, 298.0
    sp.vel = synthetic._maxwell(rng, [a[6] for a in sp.atoms], sp.temperature)
    return system.relax(sp)


CASES = [
    (5997, (40, 48, 40), 0),        # in line, line form
    (6000, (40, 48, 40), 0),        # pair kernel on the branch
    (6000, (40, 40, 40), 0),        # transforms on the branch, plane form
    (8997, (48, 48, 48), 1),        # MFMA in line
    (9000, (48, 48, 48), 1),        # MFMA: half of them before the fork
    (23558, (60, 64, 72), 0),       # pair kernel and dU/dlambda on branches
]


def _spec(atoms, grid, fft):
    sp = copy.copy(relaxed("config2") if atoms == 23558 else _water(atoms // 3))
    assert len(sp.atoms) == atoms
    sp.grid, sp.fft_mode = grid, fft
    return sp


@pytest.mark.parametrize("atoms,grid,fft", CASES)
def test_branches(atoms, grid, fft):
    sp = _spec(atoms, grid, fft)
    runs = []
    for use_graph in (True, False):
        s = system.build(sp)
        s.run_dynamics(30, freq_nrg=10, use_graph=use_graph)
        runs.append((s.positions(), s.energy(), s.lambdas()))
        if use_graph:
            s.run_energy()
            fo, do, eo, pairs = orc.forces(s.topology(), s.runparams(), s.positions(),
                                        s.lambdas() if sp.nblocks > 1 else np.ones(1))
            fg, eg = s.forces(), s.energy()
        s.close()
    print("\n[%d atoms, grid %s, fft %d] force relRMS %.2e" % (atoms, grid, fft, rel_rms(fg, fo)), flush=True)
    assert all(np.array_equal(a, b) for a, b in zip(*runs))
    assert rel_rms(fg, fo) <= 1e-5
    assert abs(eg[20] - eo[20]) <= 1e-6 * abs(eo[20])


@pytest.mark.parametrize("atoms,grid,fft", CASES)
def test_runs_of_steps_in_one_graph(atoms, grid, fft):
    """stretches of 15 and 7 plain steps between rebuilds (every 16) and
    energies (every 24), played in graphs of 8, 4, 2 and 1 steps, against the
    steps launched one by one, to the bit; twice, the second time from the
    state and graphs of the first"""
    sp = _spec(atoms, grid, fft)
    runs = []
    for use_graph in (1, 0):
        s = system.build(sp)
        s.set_domdec_frequency(16)
        s.run_energy()
        L, dev = s.L, s.device()
        if use_graph:
            assert L.bm_capture_graphs(dev) == 0
        for step in (0, 48):
            assert L.bm_dynamics(dev, step, 48, 24, use_graph) == 0
            runs.append((*system.state(s, sp.n, sp.nblocks), s.energy()))
        s.close()
    assert all(np.all(np.isfinite(a)) for a in runs[3])
    for graph, eager in ((runs[0], runs[2]), (runs[1], runs[3])):
        assert all(np.array_equal(a, b) for a, b in zip(graph, eager))
