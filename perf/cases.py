"""What is measured: molecular dynamics, batched dynamics and single-point
energies, through the blade_* / bm_* calls that a program makes.

A case is a plain dict:

  kind      "dynamics" (BladeSystem.run_dynamics), "batch" (Batch.dynamics) or
            "energy" (set_positions, run_energy and the getters)
  atoms     atoms of the system (of the largest member of a batch)
  aspect    z edge over x and y edge of the box
  sites     solute chains in TIP3P water, each carrying a lambda site of three
            substituents (0: water alone)
  chain     atoms of a chain
  soft      soft-core pairs with only dihedrals lambda-scaled (the options of
            the reference's MSLD decks), or plain
            scaling of every term (energies only: without a soft core a
            substituent's water may step into it as its lambda falls)
  elec      "pme", "fswitch" or "fshift"
  order, rcut, rswitch, fft   spline order, cutoffs, PME FFT form (0 FP32
            Stockham, 1 MFMA split BF16)
  rebuild   steps between list rebuilds
  steps     steps of one pass (dynamics and batches)
  nrg       steps between energy evaluations (0: none)
  members, smallest   systems of a batch; atoms of its smallest member (equal
            to `atoms`: lambda-replicas of one structure)

Every structure is generated and relaxed on the GPU once per process; the
seed gives each state its own origin of the periodic box, Maxwell velocities,
theta and thermostat stream.  Dynamics continue from the state the last pass
left, as a program's production loop does.
"""
import copy
import functools
import math

import numpy as np
import torch

from blade_amd import synthetic, system
from blade_amd._ffi import check

DENSITY = synthetic.WATER_DENSITY
BASE_SEED = 0xB1ADE0
# chains whose substituents do not land on their core
CHAIN_SEED = {60: 0xB1ADE007, 84: 0xB1ADE00D, 400: 0xB1ADE004, 1001: 0xB1ADE00A}


def _case(kind, atoms, **kw):
    c = dict(kind=kind, atoms=atoms, aspect=1.0, sites=0, chain=0, soft=1, elec="pme", order=6, rcut=10.0, rswitch=9.0,
             fft=0, rebuild=10, steps=0, nrg=0, members=1, smallest=atoms)
    c.update(kw)
    return c


def listed():
    return [
        # the 216-water box of the reference's test deck: the shortest step,
        # bound by launches and latency
        _case("dynamics", 648, name="water648", rcut=9.0, rswitch=8.0, steps=50),
        # a ligand in a small box with energies written every tenth step
        _case("dynamics", 4000, name="msld4000_nrg10", chain=400, steps=50, nrg=10, sites=1),
        # the headline MSLD box: 62 A, PME 64^3 order 6
        _case("dynamics", 23558, name="msld23558", chain=1001, steps=50, sites=1),
        # the settings of the reference's benchmark deck (cutoff 9/7.5 A,
        # order 4) without lambda sites
        _case("dynamics", 23559, name="deck23559", order=4, rcut=9.0, rswitch=7.5, steps=50),
        # a membrane-shaped box: unequal PME edges (no square y-z plane)
        _case("dynamics", 31116, name="slab31116", aspect=1.45, steps=40),
        # cutoff electrostatics (force switch), no PME
        _case("dynamics", 11121, name="cutoff11121", elec="fswitch", steps=50),
        # the precision form: two lambda sites, soft core, PME on the matrix cores
        _case("dynamics", 92224, name="sites92224", sites=2, chain=400, fft=1, steps=20),
        # lambda-replicas of one structure advanced together
        _case("batch", 5000, name="replicas8x5000", chain=84, members=8, steps=40, sites=1),
        # ligands of a screening run: boxes of different sizes advanced together
        _case("batch", 14003, name="mixed6", chain=84, members=6, smallest=3282, steps=40, sites=1),
        # single-point energies and forces of supplied coordinates (what a
        # host program's energy call costs), smallest, ordinary and largest
        _case("energy", 648, name="energy648", rcut=9.0, rswitch=8.0),
        _case("energy", 23558, name="energy23558", chain=1001, soft=0, sites=1),
        _case("energy", 92224, name="energy92224", sites=2, chain=400, fft=1),
    ]


def draw(rng):
    kind = rng.choice(["dynamics", "dynamics", "dynamics", "batch", "energy"])
    hi = {"dynamics": 92000, "batch": 16000, "energy": 92000}[kind]
    atoms = int(math.exp(rng.uniform(math.log(700), math.log(hi))))
    c = _case(kind, atoms)
    c["sites"] = rng.choice([0, 1, 1, 2]) if kind != "batch" else 1
    if c["sites"] == 2 and atoms < 4000:
        c["sites"] = 1
    if c["sites"]:
        c["chain"] = 60 if atoms < 2000 else rng.choice([60, 84, 400] if atoms > 8000 else [60, 84])
    c["aspect"] = rng.choice([1.0, 1.0, 1.3, 1.6]) if atoms > 6000 else 1.0
    c["elec"] = rng.choice(["pme"] * 6 + ["fswitch", "fshift"])
    c["order"] = rng.choice([4, 6, 6, 6, 8])
    c["rcut"], c["rswitch"] = (9.0, 8.0) if atoms < 1500 else rng.choice([(10.0, 9.0), (10.0, 8.5), (9.0, 7.5)])
    c["fft"] = int(c["elec"] == "pme" and atoms > 4000 and rng.random() < 0.3)
    c["rebuild"] = rng.choice([10, 10, 20])
    if kind == "batch":
        c["members"] = rng.randint(2, 8)
        c["smallest"] = atoms if rng.random() < 0.5 else max(700, int(atoms * rng.uniform(0.3, 0.9)))
    else:
        c["smallest"] = atoms
    if kind != "energy":
        # no more work than the largest listed cases
        most = (1100000 if kind == "batch" else 1500000) // sum(_sizes(c))
        c["steps"] = max(5, min(rng.randint(20, 50), most))
        c["nrg"] = rng.choice([0, 0, 10, 25]) if kind == "dynamics" else 0
    return c


# ---------------------------------------------------------------------------
# structures
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _chain(atoms):
    """a chain with one lambda site of three substituents (and one water,
    its last three atoms)"""
    return synthetic.config2(seed=CHAIN_SEED[atoms], n_water=1, n_poly=atoms, box=200.0)


def _solute(sites, chain, box):
    """`sites` chains along the box diagonal, one lambda site each: a Spec
    without water and the chains' positions"""
    if not sites:
        spec, _ = synthetic.water_box(1, box, BASE_SEED)
        spec.atoms, spec.bonds, spec.angles = [], [], []
        return spec, np.zeros((0, 3))
    one = _chain(chain)
    spec = copy.copy(one)
    spec.atoms, spec.bonds, spec.angles, spec.dihes, spec.imprs = [], [], [], [], []
    pos, block = [], []
    for k in range(sites):
        spec.atoms += one.atoms[:chain]
        for name in ("bonds", "angles", "dihes", "imprs"):
            getattr(spec, name).extend(tuple(i + k * chain for i in term) for term in getattr(one, name)
                                       if max(term) < chain)
        pos.append(one.pos[:chain] - 100.0 + np.array(box) * (k + 0.5) / sites)
        block.append(np.where(one.atom_block[:chain] > 0, one.atom_block[:chain] + 3 * k, 0))
    spec.atom_block = np.concatenate(block)
    spec.nblocks = 1 + 3 * sites
    spec.block_site = [0] + [1 + k // 3 for k in range(3 * sites)]
    spec.theta0, spec.fixed_bias = [0.0] * spec.nblocks, [0.0] * spec.nblocks
    spec.theta_mass = [0.0] + [12.0] * (3 * sites)
    return spec, np.concatenate(pos)


def _rotations(rng, n):
    q = rng.normal(size=(n, 4))
    w, x, y, z = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], axis=1).reshape(n, 3, 3)


def _mindist(p, to, box):
    """distance of each point of p to the nearest point of `to`, periodic"""
    if not len(to):
        return np.full(len(p), 1e9)
    a, b, L = (torch.as_tensor(np.asarray(v), dtype=torch.float64) for v in (p, to, box))
    out = []
    for c in a.split(4096):
        d = c[:, None, :] - b[None]
        d -= L * torch.round(d / L)
        out.append(d.square().sum(-1).amin(1).sqrt())
    return torch.cat(out).numpy()


def _solvate(spec, pos, atoms, rng):
    """TIP3P water on a lattice clear of the solute, up to `atoms` atoms"""
    L = np.array(spec.box)
    nwat = (atoms - len(pos)) // 3
    factor = 1.0
    while True:
        n1 = np.ceil(L / (L.prod() / (nwat * factor)) ** (1 / 3) - 1e-9).astype(int)
        o = (np.stack(np.meshgrid(*[np.arange(k) for k in n1], indexing="ij"), -1).reshape(-1, 3) + 0.5) * (L / n1)
        o = o[_mindist(o, pos, L) > 2.5]
        if len(o) >= nwat:
            break
        factor *= 1.05
    o = o[np.sort(rng.permutation(len(o))[:nwat])]
    half = math.radians(104.52) / 2
    h = 0.9572 * np.array([[math.sin(half), math.cos(half), 0.0], [-math.sin(half), math.cos(half), 0.0]])
    rot = _rotations(rng, nwat)
    # a few more orientations for the waters whose hydrogens face the solute
    for _ in range(12):
        hy = o[:, None, :] + np.einsum("nij,kj->nki", rot, h)
        bad = np.nonzero(_mindist(hy.reshape(-1, 3), pos, L).reshape(-1, 2).min(1) < 1.9)[0]
        if not len(bad):
            break
        rot[bad] = _rotations(rng, len(bad))
    hy = o[:, None, :] + np.einsum("nij,kj->nki", rot, h)
    base = len(pos)
    for w in range(nwat):
        b = base + 3 * w
        for nm, t, q in (("OH2", "OT", -0.834), ("H1", "HT", 0.417), ("H2", "HT", 0.417)):
            spec.atoms.append(("WAT", str(w + 1), "TIP3", nm, t, q, synthetic.WATER_TYPES[t]))
        spec.bonds += [(b, b + 1), (b, b + 2), (b + 1, b + 2)]
        spec.angles.append((b + 1, b, b + 2))
    spec.pos = np.concatenate([np.asarray(pos).reshape(-1, 3), np.concatenate([o[:, None, :], hy], 1).reshape(-1, 3)]) % L
    block = np.zeros(spec.n, dtype=np.int32)
    if spec.nblocks > 1:
        block[:base] = spec.atom_block[:base]
    spec.atom_block = block


@functools.lru_cache(maxsize=None)
def _relaxed(atoms, aspect, sites, chain, soft, elec, order, rcut, rswitch, fft):
    """the generated structure after the GPU relaxation"""
    rng = np.random.default_rng(BASE_SEED + atoms)
    a = (atoms / DENSITY / aspect) ** (1 / 3)
    box = (a, a, a * aspect)
    spec, pos = _solute(sites, chain, box)
    spec.box = box
    _solvate(spec, pos, atoms, rng)
    if sites and soft:
        spec.soft_core, spec.scale_terms = True, (0, 0, 0, 1, 0, 1)
    spec.rcut, spec.rswitch, spec.order = rcut, rswitch, order
    spec.beta = 0.34 if rcut < 10.0 else 1.0 / 3.2
    spec.elec_method = {"fswitch": 0, "pme": 1, "fshift": 2}[elec]
    spec.grid, spec.grid_space, spec.fft_mode = (-1, -1, -1), 1.0, fft
    if fft:   # the matrix-core FFT takes edges that are multiples of 16
        spec.grid = tuple(16 * math.ceil(L / 1.06 / 16) for L in box)
    spec.temperature = 298.0
    spec.vel = _velocities(spec, rng)
    return system.relax(spec)


def _velocities(spec, rng):
    m = np.array([a[6] for a in spec.atoms])[:, None]
    v = rng.normal(size=(spec.n, 3)) * np.sqrt(synthetic.KBOLTZ * spec.temperature / m)
    return v - (m * v).sum(0) / m.sum()


def _spec(case, atoms, seed):
    """one member's input: the relaxed structure with the seed's own origin,
    velocities, theta and thermostat stream"""
    base = _relaxed(atoms, case["aspect"], case["sites"], case["chain"], case["soft"], case["elec"], case["order"],
                    case["rcut"], case["rswitch"], case["fft"])
    rng = np.random.default_rng([seed, atoms])
    spec = copy.copy(base)
    spec.pos = (base.pos + rng.uniform(0.0, 1.0, 3) * np.array(base.box)) % np.array(base.box)
    spec.vel = _velocities(base, rng)
    if base.nblocks > 1:
        spec.theta0 = [0.0] + [float(t) + float(rng.normal(0.0, 0.05)) for t in base.theta0[1:]]
        spec.theta_v = None
    spec.seed = int(rng.integers(1, 1 << 62))
    spec.freq_domdec = case["rebuild"]
    return spec


def _sizes(case):
    lo, hi, m = case["smallest"], case["atoms"], case["members"]
    return [hi if m == 1 else int(round(lo * (hi / lo) ** (k / (m - 1)))) for k in range(m)]


# ---------------------------------------------------------------------------
# the measured calls
# ---------------------------------------------------------------------------
class _Batch(system.Batch):
    """closed before its members"""

    def __del__(self):
        self.close()


def prepare(case, seed):
    """built systems with their first energy evaluated, and a single system's
    step graphs captured, as a production run has them before its loop"""
    systems, specs = [], []
    for k, atoms in enumerate(_sizes(case)):
        spec = _spec(case, atoms, seed * 64 + k)
        s = system.build(spec)
        s.run_energy()
        systems.append(s)
        specs.append(spec)
    state = {"case": case, "systems": systems, "specs": specs, "step": 1}
    if case["kind"] == "energy":
        # the coordinates a host program hands over: the structure displaced
        # by what a few steps move it
        rng = np.random.default_rng([seed, 7])
        x = specs[0].pos + rng.normal(0.0, 0.01, specs[0].pos.shape)
        state["x"] = system.soa(x)
    elif case["kind"] == "batch":
        state["batch"] = _Batch(systems)
    else:
        check(systems[0].L.bm_capture_graphs(systems[0].device()), "graph capture")
    return state


def run(state):
    case, systems = state["case"], state["systems"]
    s = systems[0]
    if case["kind"] == "energy":
        s.set_positions(state["x"])
        s.run_energy()
        return {"forces": s.forces(), "terms": s.energy(), "dudl": s.dudl()}
    if case["kind"] == "batch":
        state["batch"].dynamics(state["step"], case["steps"], case["nrg"])
        state["batch"].sync()
        state["step"] += case["steps"]
    else:
        s.run_dynamics(case["steps"], freq_nrg=case["nrg"])
    out = []
    for s in systems:
        pos, vel, theta, theta_v = system.state(s, s.n, s.nblocks)
        out.append({"pos": pos, "vel": vel, "theta": theta, "theta_v": theta_v, "lambda": s.lambdas()})
    return out


def work(case):
    """bytes: positions, velocities and forces of every step read or written
    once, charges and types read once; flops: 64 a pair in the cutoff, the
    spline spread and gather, both transforms and the bonded and constraint
    arithmetic (about 500 an atom)"""
    nbytes = flops = 0.0
    steps = max(1, case["steps"])
    for n in _sizes(case):
        pairs = n * 0.5 * DENSITY * 4.0 / 3.0 * math.pi * case["rcut"] ** 3
        f = 64.0 * pairs + 500.0 * n
        if case["elec"] == "pme":
            g = n / DENSITY
            f += n * 10.0 * case["order"] ** 3 + 10.0 * g * math.log2(g)
        flops += steps * f
        nbytes += steps * n * (24.0 * (5 if case["steps"] else 2) + 16.0)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """energies: FP32 pair and grid sums carry about 1e-6 of the forces (the
    matrix-core FFT's split BF16 products up to 8e-6).  Trajectories amplify
    the forces' rounding: with the pair sums in another order the velocities
    differ by 1e-6 to 2e-6 of their norm after 50 steps and by 6e-6 to 1.1e-5
    after 100 (a second pass), single ones by up to 100 times that of their
    root mean square"""
    if case["kind"] == "energy":
        return {"rel": 3e-5, "max": 1e-3} if case["fft"] else {"rel": 1e-5, "max": 5e-4}
    rel = 4e-6 * math.exp(0.05 * case["steps"])
    return {"rel": rel, "max": 100.0 * rel}


# ---------------------------------------------------------------------------
# 64-bit reference of an energy call, in plain torch
# ---------------------------------------------------------------------------
KE = 332.0716


def _pair_energy(c, qq, c12, c6, r, shift14=False, e14=None):
    """energy of pairs at distance r < rcut; shift14: the 1-4 form of the
    force-switched van der Waals energy (and e14 scaling the charges)"""
    rc, rs = c["rcut"], c["rswitch"]
    if c["elec"] == "pme":
        beta = 0.34 if rc < 10.0 else 1.0 / 3.2
        e = KE * qq * (torch.erfc(beta * r) + (0.0 if e14 is None else e14 - 1.0)) / r
    elif c["elec"] == "fswitch":
        of, on = rc * rc, rs * rs
        g = (of - on) ** -3
        A, B, C, D = of * of * (of - 3 * on) * g, 6 * of * on * g, -(on + of) * g, 0.4 * g
        dvc = 8 * (on * of * (rc - rs) - (of * of * rc - on * on * rs) / 5) * g
        inner = 1 / r + dvc
        outer = A * (1 / r - 1 / rc) + B * (rc - r) + C * (of * rc - r ** 3) + D * (of * of * rc - r ** 5)
        e = KE * qq * (1.0 if e14 is None else e14) * torch.where(r <= rs, inner, outer)
    else:
        e = KE * qq * (1.0 if e14 is None else e14) * (1 / r - 2 / rc + r / rc ** 2)
    r3, r6 = r ** -3, r ** -6
    k6, k12 = rc ** 3 / (rc ** 3 - rs ** 3), rc ** 6 / (rc ** 6 - rs ** 6)
    s6, s12 = (rc ** -6, rc ** -12) if shift14 else ((rc * rs) ** -3, (rc * rs) ** -6)
    rep = torch.where(r < rs, r6 * r6 - s12, k12 * (r6 - rc ** -6) ** 2)
    att = torch.where(r < rs, r6 - s6, k6 * (r3 - rc ** -3) ** 2)
    return e + c12 * rep - c6 * att


def _spline(order, u):
    """weights of the order points around fraction u, [..., order]: point t
    takes M_order(u + order - 1 - t)"""
    a = [torch.ones_like(u)]
    for m in range(2, order + 1):
        b = a + [torch.zeros_like(u)]
        a = [((u + k) * b[k] + ((m - u - k) * b[k - 1] if k else 0.0)) / (m - 1) for k in range(m)]
    return torch.stack(a[::-1], -1)


def exact(case, seed):
    """a trajectory has no value of its own to state (its noise is the
    library's random stream); an energy call is evaluated in 64 bits by
    automatic differentiation of the energy"""
    if case["kind"] != "energy":
        return None
    state = prepare(case, seed)
    s, spec, c = state["systems"][0], state["specs"][0], case
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f64 = dict(dtype=torch.float64, device=dev)
    t, rp = s.topology().contents, s.runparams().contents
    n, nl = t.n_atoms, max(1, t.n_blocks)

    def arr(name, count, width=1):
        a = t.array(name, count, width)
        return torch.as_tensor(a, device=dev).long() if a.dtype == np.int32 else torch.as_tensor(a, **f64)

    L = torch.tensor(list(rp.box), **f64)
    x = torch.as_tensor(state["x"].reshape(3, n).T.copy(), **f64).requires_grad_()
    lam = torch.ones(nl, **f64)
    site_of = torch.tensor(spec.block_site, device=dev)
    theta = torch.tensor(spec.theta0, **f64)
    for q in range(1, int(site_of.max()) + 1):
        lam[site_of == q] = torch.softmax(spec.fnex * torch.sin(theta[site_of == q]), 0)
    lam.requires_grad_()
    block = arr("site_block", n) & 0xFFFF
    q, typ = arr("charge", n), arr("type_idx", n)
    c12, c6 = arr("vdw_c12", t.n_types ** 2), arr("vdw_c6", t.n_types ** 2)
    terms = torch.zeros(23, **f64)

    def add(index, e, keep=False):
        terms[index] += float(e.detach())
        if e.requires_grad:
            e.backward(retain_graph=keep)

    def image(d):
        return d - L * torch.round(d.detach() / L)

    def scale(sb):
        b = sb & 0xFFFF
        one = torch.ones(len(b), **f64)
        l0 = torch.where(b[:, 0] > 0, lam[b[:, 0]], one)
        return l0 * torch.where((b[:, 0] > 0) & (b[:, 1] > 0), lam[b[:, 1]], one)

    # nonbonded pairs: those within the cutoff found row by row, each once
    ex = arr("excl_idx", t.n_excl, 2)
    key = torch.sort(torch.cat([ex[:, 0] * n + ex[:, 1], ex[:, 1] * n + ex[:, 0]]))[0]
    soft = bool(rp.soft_core) and nl > 1
    rows = max(1, int(1.0e8 // n))
    for i0 in range(0, n, rows):
        with torch.no_grad():
            d2 = 0.0
            for k in range(3):
                d = x[i0:i0 + rows, k][:, None] - x[None, i0:, k]
                d2 = d2 + (d - L[k] * torch.round(d / L[k])).square()
            i, j = torch.nonzero(d2 < rp.rcut ** 2, as_tuple=True)
            i, j = i + i0, j + i0
            keep = i < j
            i, j = i[keep], j[keep]
            if len(key):
                at = torch.searchsorted(key, i * n + j).clamp(max=len(key) - 1)
                keep = key[at] != i * n + j
                i, j = i[keep], j[keep]
            bi, bj = block[i], block[j]
            same = site_of[bi] == site_of[bj]
            keep = ~(same & (bi != bj))
            i, j, bi, bj, same = i[keep], j[keep], bi[keep], bj[keep], same[keep]
        r = image(x[i] - x[j]).square().sum(-1).sqrt()
        w = torch.where(same, lam[bi], lam[bi] * lam[bj])
        if soft:
            rsoft = 4.0 * (1.0 - w)
            inside = ((bi > 0) | (bj > 0)) & (r.detach() < rsoft.detach())
            ratio = r / torch.where(inside, rsoft, torch.ones_like(rsoft))
            r = torch.where(inside, ((1.0 - 0.5 * ratio) * ratio ** 3 + 0.5) * rsoft, r)
        ti = typ[i] * t.n_types + typ[j]
        add(7, (w * _pair_energy(c, q[i] * q[j], c12[ti], c6[ti], r)).sum())
    # bonded terms
    idx = arr("bond_idx", t.n_bonds, 2)
    r = image(x[idx[:, 0]] - x[idx[:, 1]]).square().sum(-1).sqrt()
    e = 0.5 * arr("bond_kb", t.n_bonds) * (r - arr("bond_b0", t.n_bonds)) ** 2 * scale(arr("bond_sb", t.n_bonds, 2))
    terms[2] += float(e[t.n_bonds12:].detach().sum())
    terms[0] -= float(e[t.n_bonds12:].detach().sum())
    add(0, e.sum())
    if t.n_angles:
        idx = arr("angle_idx", t.n_angles, 3)
        a, b = image(x[idx[:, 0]] - x[idx[:, 1]]), image(x[idx[:, 2]] - x[idx[:, 1]])
        th = torch.atan2(torch.linalg.cross(a, b).square().sum(-1).sqrt(), (a * b).sum(-1))
        e = 0.5 * arr("angle_k", t.n_angles) * (th - arr("angle_t0", t.n_angles)) ** 2
        add(1, (e * scale(arr("angle_sb", t.n_angles, 2))).sum())
    for name, count, index in (("dihe", t.n_dihes, 3), ("impr", t.n_imprs, 4)):
        if not count:
            continue
        idx = arr(name + "_idx", count, 4)
        a, b, d = (image(x[idx[:, k]] - x[idx[:, k + 1]]) for k in range(3))
        m, v = torch.linalg.cross(a, b), torch.linalg.cross(b, d)
        # sin(phi) = -|b| a.(b x d) / |m||v|: positive phi for a negative triple product
        phi = torch.atan2(-b.square().sum(-1).sqrt() * (a * v).sum(-1), (m * v).sum(-1))
        k, mult, d0 = arr(name + "_k", count), arr(name + "_n", count), arr(name + "_d0", count)
        dp = phi - d0
        dp = dp - 2 * math.pi * torch.floor((dp.detach() + math.pi) / (2 * math.pi))
        periodic = k * (torch.cos(mult * phi - d0) + 1.0)
        e = periodic if index == 3 else torch.where(mult > 0, periodic, 0.5 * k * dp ** 2)
        add(index, (e * scale(arr(name + "_sb", count, 2))).sum())
    if t.n_nb14:
        idx = arr("nb14_idx", t.n_nb14, 2)
        r = image(x[idx[:, 0]] - x[idx[:, 1]]).square().sum(-1).sqrt()
        e = _pair_energy(c, arr("nb14_qq", t.n_nb14), arr("nb14_c12", t.n_nb14), arr("nb14_c6", t.n_nb14), r, True,
                         arr("nb14_e14fac", t.n_nb14))
        add(6, torch.where(r < rp.rcut, e * scale(arr("nb14_sb", t.n_nb14, 2)), torch.zeros_like(r)).sum())
    if case["elec"] == "pme":
        beta = rp.beta_ewald
        if t.n_nbex:
            idx = arr("nbex_idx", t.n_nbex, 2)
            r = image(x[idx[:, 0]] - x[idx[:, 1]]).square().sum(-1).sqrt()
            e = -KE * arr("nbex_qq", t.n_nbex) * torch.erf(beta * r) / r
            add(10, (e * scale(arr("nbex_sb", t.n_nbex, 2))).sum())
        lq = torch.where(block > 0, lam[block], torch.ones(n, **f64)) * q
        add(9, -beta * KE / math.sqrt(math.pi) * lq.square().sum())
        # smooth PME: spread, structure factor, energy sum over wavevectors
        K, order = list(rp.grid), rp.order
        lq = torch.where(block > 0, lam[block], torch.ones(n, **f64)) * q
        grid = torch.zeros(K[0] * K[1] * K[2], **f64)
        w, at = [], []
        for k in range(3):
            u = x[:, k] * (K[k] / L[k])
            u0 = torch.floor(u.detach())
            w.append(_spline(order, u - u0))
            at.append((u0.long()[:, None] + torch.arange(order, device=dev)) % K[k])
        cell = (at[0][:, :, None, None] * K[1] + at[1][:, None, :, None]) * K[2] + at[2][:, None, None, :]
        value = lq[:, None, None, None] * w[0][:, :, None, None] * w[1][:, None, :, None] * w[2][:, None, None, :]
        S = torch.fft.fftn(grid.index_add(0, cell.reshape(-1), value.reshape(-1)).reshape(K))
        fac = torch.full(K, 0.5 * KE / math.pi / float(L.prod()), **f64)
        m2 = torch.zeros(K, **f64)
        whole = _spline(order, torch.zeros(1, **f64))[0]   # M_order at the integers order-1 .. 0
        for k in range(3):
            m = torch.arange(K[k], **f64)
            ang = 2 * math.pi * m[:, None] * torch.arange(order, **f64) / K[k]
            mod = 1.0 / ((whole * torch.cos(ang)).sum(-1) ** 2 + (whole * torch.sin(ang)).sum(-1) ** 2)
            shape = [-1 if d == k else 1 for d in range(3)]
            fac = fac * mod.reshape(shape)
            m2 = m2 + (torch.where(2 * m <= K[k], m, m - K[k]) / L[k]).square().reshape(shape)
        m2[0, 0, 0] = 1.0
        fac = fac * torch.exp(-math.pi ** 2 / beta ** 2 * m2) / m2
        fac[0, 0, 0] = 0.0
        add(8, (fac * (S.real.square() + S.imag.square())).sum())
    terms[20] = terms[:20].sum()
    terms[22] = terms[20]
    dudl = torch.zeros(nl, **f64) if lam.grad is None else lam.grad.clone()
    dudl[0] = 0.0
    return {"forces": x.grad.T.reshape(-1).cpu().numpy(), "terms": terms.cpu().numpy(), "dudl": dudl.cpu().numpy()}
