"""The workloads this engine is measured on, through its public entry points.

Seven kinds of calls, over the sizes and options of the repository's own
benchmark, configurations and tests:

  water    explicit solvent MD (pdgpu_md): TIP3P boxes, force-switched Coulomb,
           velocity Verlet, Beeman or Langevin, with or without the
           Berendsen thermostat, the list rebuilt every 10 steps;
  vacuum   MD of one AMBER99 chain with the nonbonded list and no box, energy- or
           force-switched;
  gb       implicit-solvent (GB/SA) Langevin MD of one AMBER99 chain;
  batch    the same for many chains of uneven length in one batch, or for the
           replicas of one chain on a temperature ladder;
  point    forces and energies of one snapshot of a water box (a rerun, or the
           force component of a host program): new list, one evaluation;
  list     the neighbour list alone, handed to host force fields in PD's packed form;
  mc       Monte Carlo moves of single molecules (pdgpu_energy_update).

MD passes of one engine start from the stored snapshot of the state, so every
pass does the same work; a batch carries its trajectories on from pass to pass.
exact() evaluates the same physics in 64 bits with plain torch.
"""
import functools
import math

import numpy as np
import torch

from pd_amd import engine as G
from pd_amd import forcefield as F
from pd_amd import systems as S

# PD's constants (SI), and the units the formulas below work in: kcal/mol, A
NA, KB, ANG = 6.0221418e23, 1.38065e-23, 1e-10
KCAL = 4184.0 / NA                                   # J per molecule
ECONV = 1.60217645e-19 ** 2 / (math.pi * 4.0 * 8.854187817e-12 * ANG) / KCAL
JM = KCAL / ANG                                      # kcal/mol/A -> J/m
MANY = 1 << 30                                       # MolecularDynamics::Steps: no pass holds the last step


# ---- the cases -------------------------------------------------------------------------

def listed():
    return [
        # a 20-residue chain in vacuum, 12 A cutoff: the smallest runs, where launches count
        dict(name="vacuum_20", kind="vacuum", residues=20, cutoff=12.0, inner=10.0, elec="energy", integrator="verlet",
             thermostat=False, fs=1.0, steps=50),
        # a 512-water box: set-up and test runs of a solvent protocol
        dict(name="water_1536", kind="water", waters=512, nx=1, ny=1, nz=1, cutoff=10.0, inner=8.0, elec="force",
             integrator="verlet", thermostat=False, fs=1.0, steps=50),
        # an NVT box of the size of a small solvated protein
        dict(name="water_12288_nvt", kind="water", waters=512, nx=2, ny=2, nz=2, cutoff=10.0, inner=8.0, elec="force",
             integrator="beeman", thermostat=True, fs=1.0, steps=40),
        # the explicit-solvent benchmark: 98,304 atoms, NVE Beeman at 1 fs
        dict(name="water_98304", kind="water", waters=512, nx=4, ny=4, nz=4, cutoff=10.0, inner=8.0, elec="force",
             integrator="beeman", thermostat=False, fs=1.0, steps=40),
        # a snapshot of the same box scored on its own
        dict(name="point_98304", kind="point", waters=512, nx=4, ny=4, nz=4, cutoff=10.0, inner=8.0, elec="force"),
        # the list handed to host force fields after a rebuild
        dict(name="list_12288", kind="list", waters=512, nx=2, ny=2, nz=2, cutoff=10.0, inner=8.0, elec="force"),
        # Monte Carlo trial moves of single waters
        dict(name="mc_1536", kind="mc", waters=512, nx=1, ny=1, nz=1, cutoff=10.0, inner=8.0, elec="force", moves=10),
        # a small chain in implicit solvent with PD's default cutoffs
        dict(name="gb_20", kind="gb", residues=20, all_pairs=False, fs=2.0, steps=20),
        # the implicit-solvent benchmark: one 300-residue chain, all pairs
        dict(name="gb_300", kind="gb", residues=300, all_pairs=True, fs=2.0, steps=20),
        # 64 replicas of a 60-residue chain on a 300-500 K ladder, between two exchanges
        dict(name="replicas_64", kind="batch", systems=64, shortest=60, longest=60, ladder=True, all_pairs=True,
             fs=2.0, steps=15),
        # 256 chains of 20-120 residues in one batch
        dict(name="batch_256", kind="batch", systems=256, shortest=20, longest=120, ladder=False, all_pairs=True,
             fs=2.0, steps=15),
    ]


def draw(rng):
    """One more case of the same ranges; no larger than the largest listed one of its kind."""
    kind = rng.choice(["water", "water", "vacuum", "gb", "gb", "batch", "batch", "point", "list", "mc"])

    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if kind == "gb":
        return dict(kind=kind, residues=spread(20, 300), all_pairs=rng.random() < 0.6, fs=rng.choice([1.0, 2.0]),
                    steps=rng.randint(10, 20))
    if kind == "batch":
        ladder = rng.random() < 0.4
        systems = spread(8, 64 if ladder else 256)
        lo = rng.randint(20, 60)
        return dict(kind=kind, systems=systems, shortest=lo, longest=lo if ladder else rng.randint(lo + 7, 120),
                    ladder=ladder, all_pairs=rng.random() < 0.8, fs=2.0, steps=rng.choice([10, 15]))
    cut = rng.choice([9.0, 10.0, 10.0])
    nb = dict(cutoff=cut, inner=cut - rng.choice([1.0, 2.0]), elec="force")
    if kind == "vacuum":
        nb["elec"] = rng.choice(["force", "energy", "energy"])
        return dict(kind=kind, residues=spread(20, 120), **nb, integrator=rng.choice(["verlet", "langevin"]),
                    thermostat=False, fs=1.0, steps=rng.randint(20, 50))
    tiles = {"water": 64, "point": 64, "list": 8, "mc": 8}[kind]
    n = 1 << rng.randint(0, tiles.bit_length() - 1)
    nx = min(n, rng.choice([1, 2, 4]))
    ny = min(n // nx, 4)
    box = dict(waters=rng.randint(343, 512), nx=nx, ny=ny, nz=min(n // nx // ny, 8))
    if kind == "water":
        integ = rng.choice(["verlet", "beeman", "langevin"])
        return dict(kind=kind, **box, **nb, integrator=integ, fs=1.0, steps=rng.randint(20, 40),
                    thermostat=integ != "langevin" and rng.random() < 0.4)
    return dict(kind=kind, **box, **nb, **(dict(moves=rng.randint(4, 12)) if kind == "mc" else {}))


# ---- what a user's program has in hand ---------------------------------------------------

PADDING, UPDATE, TEMP, FRICTION, TAU, SASA_EVERY, ASP = 2.0, 10, 300.0, 1e12, 100e-15, 5, 0.005


def nb_kw(case):
    c, i = case["cutoff"], case["inner"]
    return dict(Cutoff=c, InnerCutoff=i, VdwCutoff=c, VdwInnerCutoff=i, ForceSwitch=int(case["elec"] == "force"),
                EnergySwitch=int(case["elec"] == "energy"))


def gb_kw(case):
    kw = dict(DielectricSolvent=78.5, Vdw14Scaling=0.5, Elec14Scaling=0.83333)
    if case["all_pairs"]:
        kw.update(Cutoff=999.0, InnerCutoff=999.0, VdwCutoff=999.0, VdwInnerCutoff=999.0, GbsaStillCutoff=999.0)
    return kw


@functools.lru_cache(maxsize=64)
def chain(residues):
    """A random-sequence AMBER99 chain, its close contacts eased by capped
    steepest-descent steps, coordinates to 1e-4 A."""
    s = F.random_peptide(residues, 1000 + residues)
    ref = Reference(s, nb=dict(Cutoff=999.0, InnerCutoff=999.0, VdwCutoff=999.0, VdwInnerCutoff=999.0,
                               ForceSwitch=0, EnergySwitch=0))
    x = torch.tensor(s.pos)
    for _ in range(60):
        x = descend(ref, x)
    s.pos = np.round(x.numpy(), 4)
    return s


@functools.lru_cache(maxsize=16)
def water(waters):
    """A cubic TIP3P box at 1 g/cm^3, quenched from the lattice the same way."""
    s = S.water_box(waters, seed=17)
    ref = Reference(s, nb=dict(Cutoff=9.0, InnerCutoff=8.0, VdwCutoff=9.0, VdwInnerCutoff=8.0, ForceSwitch=1))
    x = torch.tensor(s.pos)
    for _ in range(120):
        x = descend(ref, x)
    s.pos = np.round(x.numpy(), 4)
    return s


def descend(ref, x):
    f = ref.forces(x)[0]
    step = 0.002 * f
    return x + step * (0.05 / step.norm(dim=1).clamp_min(0.05))[:, None]


def shake(rng, pos, mass, temp):
    """Thermal displacements and Maxwell-Boltzmann velocities (m/s)."""
    x = pos + 0.03 * rng.standard_normal(pos.shape) * np.sqrt(1.66e-27 / mass)[:, None]
    return x, rng.standard_normal(pos.shape) * np.sqrt(KB * temp / mass)[:, None]


@functools.lru_cache(maxsize=16)
def tiled(waters, nx, ny, nz):
    """The quenched box repeated nx x ny x nz times: one system of nx*ny*nz*waters waters."""
    unit = water(waters)
    if nx * ny * nz == 1:
        return unit
    s = S.water_box(waters * nx * ny * nz, seed=1)
    s.box = unit.box * np.array([nx, ny, nz], dtype=np.float64)
    at = np.stack(np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij"), -1).reshape(-1, 3)
    at = (at - (np.array([nx, ny, nz]) - 1) / 2.0) * unit.box
    s.pos = (unit.pos[None] + at[:, None]).reshape(-1, 3)
    return s


def system(case):
    return chain(case["residues"]) if "residues" in case else tiled(case["waters"], case["nx"], case["ny"], case["nz"])


def inputs(case, seed):
    """[(system, positions, velocities, temperature)] of a case, from the seed alone."""
    rng = np.random.default_rng([seed, 77])
    if case["kind"] == "list":  # one conformation, drifted through the box: as many pairs for every seed
        s = system(case)
        x, v = shake(np.random.default_rng(78), s.pos, s.mass, TEMP)
        return [(s, x + np.round(rng.uniform(-0.5, 0.5, 3) * s.box, 3), v, TEMP)]
    if case["kind"] != "batch":
        s = system(case)
        return [(s, *shake(rng, s.pos, s.mass, TEMP), TEMP)]
    n, lo, hi = case["systems"], case["shortest"], case["longest"]
    out = []
    for k in range(n):  # up to eight chain lengths, each system a conformer of its own
        s = chain(lo + (hi - lo) * (k % 8) // 7)
        t = TEMP * (500.0 / 300.0) ** (k / max(n - 1, 1)) if case["ladder"] else TEMP
        x, v = shake(rng, s.pos @ S.random_rotation(rng).T, s.mass, t)
        out.append((s, x, v, t))
    return out


def moved(case, seed, x):
    """The positions after each Monte Carlo move: one molecule shifted and turned."""
    rng = np.random.default_rng([seed, 78])
    out = [x]
    for _ in range(case["moves"]):
        x = x.copy()
        m = slice(*(3 * rng.integers(0, len(x) // 3) + np.array([0, 3])))
        turn = np.linalg.qr(np.eye(3) + 0.1 * rng.standard_normal((3, 3)))[0]
        turn *= np.sign(np.diag(turn))[None]
        c = x[m].mean(axis=0)
        x[m] = (x[m] - c) @ turn.T + c + rng.uniform(-0.1, 0.1, 3)
        out.append(x)
    return out


def gb_engine(case, s, x, v):
    e = G.engine_for(s, None, bonded=True)
    e.setup_gb(G.gb_params(**gb_kw(case)), s.gbrad, s.cov)
    use, rad, p = F.lcpo_params_ff(s)
    e.setup_lcpo(G.LCPOParams(GlobalASP=ASP, UpdateSasa=SASA_EVERY), rad, p, use)
    e.set_positions(x)
    e.set_velocities(v)
    return e


def md_params(case, seed):
    gb = case["kind"] in ("gb", "batch")
    integ = {"verlet": G.PDGPU_VELOCITY_VERLET, "beeman": G.PDGPU_BEEMAN,
             "langevin": G.PDGPU_LANGEVIN}[case.get("integrator", "langevin")]
    return G.MDParams(integrator=integ, components=G.PDGPU_BONDED | (G.PDGPU_GB | G.PDGPU_SASA if gb else G.PDGPU_NONBONDED),
                      timestep=case["fs"] * 1e-15, temperature=TEMP, fric_coeff=FRICTION,
                      update_nlist=0 if gb else UPDATE, step_offset=0, total_steps=MANY, seed=seed % 1000003,
                      noise_stream=0, thermostat=G.PDGPU_BERENDSEN if case.get("thermostat") else G.PDGPU_NO_THERMOSTAT,
                      berendsen_tau=TAU)


def prepare(case, seed):
    kind, given = case["kind"], inputs(case, seed)
    s, x, v, _ = given[0]
    state = dict(kind=kind, x=x, v=v)
    if kind in ("water", "vacuum", "gb", "batch"):
        state.update(md=md_params(case, seed), steps=case["steps"])
    if kind == "batch":
        engines = [gb_engine(case, s, x, v) for s, x, v, _ in given]
        state["batch"] = b = G.Batch(engines)
        b.set_temperatures([t for *_, t in given])
        return state
    if kind == "gb":
        state["engine"] = gb_engine(case, s, x, v)
        return state
    state["engine"] = e = G.engine_for(s, G.nb_params(**nb_kw(case)), padding=PADDING, bonded=kind != "mc")
    e.set_positions(x)
    e.set_velocities(v)
    if kind == "mc":
        state["moves"] = moved(case, seed, x)
        e.build_list()
    return state


def run(state):
    kind = state["kind"]
    if kind == "batch":
        b = state["batch"]
        epot, ekin = b.md(state["md"], state["steps"])
        state["md"].step_offset += state["steps"]
        return dict(epot=epot, ekin=ekin, pos=np.concatenate([b.get_positions(k) for k in range(b.nsys)]))
    e = state["engine"]
    if kind == "mc":
        out = []
        for x in state["moves"]:
            e.set_positions(x)
            en = e.energy_update()
            out.append((en["epot"], en["epot_vdw"], en["epot_elec"]))
        return dict(energies=np.array(out))
    e.set_positions(state["x"])
    if kind == "list":
        e.build_list()
        counts, packed = e.get_pairs()
        return dict(counts=counts, packed=packed)
    if kind == "point":
        e.build_list()
        f, en = e.compute(G.PDGPU_NONBONDED | G.PDGPU_BONDED)
        return dict(forces=f, energies=np.array([en[k] for k in G.ENERGY_FIELDS]))
    e.set_velocities(state["v"])
    epot, ekin = e.md(state["md"], state["steps"])
    return dict(epot=epot, ekin=ekin, pos=e.get_positions(), vel=e.get_velocities())


def work(case):
    """Bytes: positions, velocities and forces of each step once, and the list's entries once
    where it is the result.  FLOP: 60 per pair within the cutoff, 174 per GB pair (three passes)."""
    kind = case["kind"]
    steps = case.get("steps", 1)
    if kind in ("gb", "batch"):
        if kind == "gb":
            sizes = [16.4 * case["residues"]]
        else:
            sizes = [16.4 * (case["shortest"] + (case["longest"] - case["shortest"]) * (k % 8) // 7)
                     for k in range(case["systems"])]
        n = sum(sizes)
        pairs = sum(m * m / 2 if case["all_pairs"] else min(m * m / 2, 160.0 * m) for m in sizes)
        return {"bytes": steps * n * 144.0, "flops": steps * (pairs * 174.0 + 300.0 * n)}
    n = 3.0 * case["waters"] * case["nx"] * case["ny"] * case["nz"] if "waters" in case else 16.4 * case["residues"]

    def pairs_to(r):
        return n * min(n / 2, 0.5 * 0.1003 * 4.19 * r ** 3)
    if kind == "list":
        return {"bytes": n * 24.0 + 4.0 * (n + pairs_to(case["cutoff"] + PADDING)), "flops": 0.0}
    if kind == "mc":
        near = 2 * 3 * 2 * pairs_to(case["cutoff"]) / n
        return {"bytes": case["moves"] * n * 24.0, "flops": 60.0 * (pairs_to(case["cutoff"]) + case["moves"] * near)}
    per = n * (48.0 if kind == "point" else 144.0)
    return {"bytes": steps * per, "flops": steps * (60.0 * pairs_to(case["cutoff"]) + 100.0 * n)}


# ---- the same physics in 64 bits ----------------------------------------------------------

def device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def bond_orders(s):
    """(n, n) bond order of each pair: 1 (1-2), 2 (1-3), 3 (1-4), else 7."""
    bo = np.full((s.n, s.n), 7, dtype=np.int8)
    for order, (off, idx) in ((3, ("off14", "idx14")), (2, ("off13", "idx13")), (1, ("off12", "idx12"))):
        i = np.repeat(np.arange(s.n), np.diff(s.cov[off]))
        bo[i, s.cov[idx]] = order
        bo[s.cov[idx], i] = order
    return bo


class Reference:
    """Forces (kcal/mol/A) and energies (kcal/mol) of one system, or of several conformers of it at once."""

    def __init__(self, s, nb=None, gb=None, lcpo=False):
        self.s, self.dev = s, device()
        t = functools.partial(torch.tensor, dtype=torch.float64, device=self.dev)
        self.eps, self.rad, self.q = t(s.epsilon / math.sqrt(KCAL)), t(s.radius), t(s.charge)
        self.nb = G.nb_params(**nb) if nb else None
        self.gb = G.gb_params(**gb) if gb else None
        self.lcpo = lcpo
        # a water box goes cell by cell (the molecules are its only bonded partners), a chain all pairs
        self.cells = s.box is not None
        if not self.cells:
            bo = torch.tensor(bond_orders(s), device=self.dev)
            self.on = (bo >= 3) & ~torch.eye(s.n, dtype=torch.bool, device=self.dev)
            self.is14 = (bo == 3).double()
        if self.gb:
            self.gb_fixed()
        if lcpo:
            use, rad, p = F.lcpo_params_ff(s)
            self.heavy = torch.tensor(np.nonzero(use)[0], device=self.dev)
            self.lr, self.lp = t(rad + 1.4)[self.heavy], t(p)[self.heavy]

    # bonds, angles, torsions: autograd on the host
    def bonded(self, x):
        s = self.s
        x = x.cpu().detach().requires_grad_()
        t = torch.tensor

        def arm(i, j):
            return x[..., t(i).long(), :] - x[..., t(j).long(), :]
        d = arm(s.bonds[:, 0], s.bonds[:, 1]).norm(dim=-1)
        e = [(t(s.bond_k / KCAL) * (d - t(s.bond_l)) ** 2).sum(-1)]
        if len(s.angles):
            u, v = arm(s.angles[:, 0], s.angles[:, 1]), arm(s.angles[:, 2], s.angles[:, 1])
            th = torch.atan2(torch.linalg.cross(u, v).norm(dim=-1), (u * v).sum(-1))
            e.append((t(s.angle_k / KCAL) * (th - t(s.angle_t0)) ** 2).sum(-1))
        else:
            e.append(torch.zeros_like(e[0]))
        if len(s.torsions):
            a, b, c = (arm(s.torsions[:, k], s.torsions[:, k + 1]) for k in range(3))
            n1, n2 = torch.linalg.cross(a, b), torch.linalg.cross(b, c)
            phi = -torch.atan2((torch.linalg.cross(b, n1) * n2).sum(-1) / b.norm(dim=-1), (n1 * n2).sum(-1))
            live = t(np.arange(4)[None] < np.asarray(s.tor_terms)[:, None])
            k, n, g = t(s.tor_vn / KCAL), t(s.tor_n), t(s.tor_gamma)
            diff = phi[..., None] - g
            diff = torch.where(diff < -math.pi, diff + 2 * math.pi, torch.where(diff > math.pi, diff - 2 * math.pi, diff))
            term = torch.where(n > 0, k * (1 + torch.cos(n * phi[..., None] + g)), k * diff ** 2)
            e.append(torch.where(live, term, torch.zeros_like(term)).sum((-1, -2)))
        else:
            e.append(torch.zeros_like(e[0]))
        f, = torch.autograd.grad(sum(v.sum() for v in e), x)
        vir = None
        if self.s.box is not None:  # bonds only enter PD's virial
            u = arm(s.bonds[:, 0], s.bonds[:, 1]).detach().norm(dim=-1)
            vir = (2 * t(s.bond_k / KCAL) * (u - t(s.bond_l)) * u).sum(-1)
        return -f.to(self.dev), [v.detach().to(self.dev) for v in e], vir

    def scaled14(self, p):
        return 1 + (p.Vdw14Scaling - 1) * self.is14, 1 + (p.Elec14Scaling - 1) * self.is14

    @staticmethod
    def switch(r, inner, cut):
        if not cut > inner:
            return torch.ones_like(r)
        t = (r - inner).clamp_min(0.0) / (cut - inner)
        return (1 - t * t) ** 2

    def lj(self, r, eps, radius, inner, cut):
        b = (radius / r) ** 6
        return eps * (b * b - 2 * b) * self.switch(r, inner, cut) * (r < cut)

    def coulomb(self, r, qq):
        """The listed pairs' Coulomb term: plain, energy-switched or force-switched."""
        p = self.nb
        c, i = p.Cutoff, p.InnerCutoff
        if p.ForceSwitch:
            sa = 1.0 / (c * c - i * i) ** 3
            co = (-(c ** 6 - 3 * c ** 4 * i * i), 6 * c * c * i * i, -(c * c + i * i), 0.4)

            def poly(r):
                return sa * (co[0] / r + co[1] * r + co[2] * r ** 3 + co[3] * r ** 5)
            e = torch.where(r <= i, 1 / r - (1 / i + poly(i) - poly(c)), poly(c) - poly(r))
        else:
            e = 1 / r * (self.switch(r, i, c) if p.EnergySwitch else 1.0)
        return qq * e * (r <= c)

    def pairs(self, d, on, eps, radius, qq):
        """Energies and forces of the left atoms of the displacements d (..., i, j, 3), each pair seen from both sides."""
        r = torch.where(on, d.pow(2).sum(-1).sqrt(), 1e3).requires_grad_()
        p = self.nb
        ev = self.lj(r, eps, radius, p.VdwInnerCutoff, p.VdwCutoff)
        ee = self.coulomb(r, qq)
        g, = torch.autograd.grad((ev + ee).sum(), r)
        r = r.detach()
        f = -(torch.where(on, g / r, 0.0)[..., None] * d).sum(-2)
        return f, 0.5 * ev.detach().sum((-1, -2)), 0.5 * ee.detach().sum((-1, -2)), 0.5 * torch.where(on, g * r, 0.0).sum((-1, -2))

    def nonbonded(self, x):
        q = self.q * math.sqrt(ECONV / self.nb.Dielectric)
        if not self.cells:
            d = x[..., :, None, :] - x[..., None, :, :]
            s14, e14 = self.scaled14(self.nb)
            return self.pairs(d, self.on, s14 * self.eps[:, None] * self.eps[None], self.rad[:, None] + self.rad[None],
                              e14 * q[:, None] * q[None])
        # water: cells at least a cutoff wide, each against its neighbours
        box = torch.tensor(self.s.box, device=self.dev)
        m = [max(1, int(v // self.nb.Cutoff)) for v in self.s.box]
        n = torch.tensor(m, device=self.dev)
        w = x - box * torch.floor(x / box + 0.5)
        at = torch.minimum(((w / box + 0.5) * n).long(), n - 1)
        cell = (at[:, 0] * m[1] + at[:, 1]) * m[2] + at[:, 2]
        order = torch.argsort(cell, stable=True)
        count = torch.bincount(cell, minlength=m[0] * m[1] * m[2])
        slot = torch.empty_like(order)
        slot[order] = torch.arange(len(order), device=self.dev) - (torch.cumsum(count, 0) - count)[cell[order]]
        table = torch.full((len(count), int(count.max())), -1, device=self.dev)
        table[cell, slot] = torch.arange(len(x), device=self.dev)
        f = torch.zeros_like(x)
        total = torch.zeros(3, dtype=torch.float64, device=self.dev)
        near = [sorted({(k + o) % c for o in (-1, 0, 1)}) for c in m for k in range(c)]
        near = [near[:m[0]], near[m[0]:m[0] + m[1]], near[m[0] + m[1]:]]
        for c in range(len(count)):
            i = table[c][table[c] >= 0]
            a, b, e = c // (m[1] * m[2]), c // m[2] % m[1], c % m[2]
            others = [(u * m[1] + v) * m[2] + k for u in near[0][a] for v in near[1][b] for k in near[2][e]]
            j = table[others].reshape(-1)
            j = j[j >= 0]
            d = x[i][:, None] - x[j][None]
            d = d - box * torch.round(d / box)
            on = (d.pow(2).sum(-1) <= self.nb.Cutoff ** 2) & (i[:, None] // 3 != j[None] // 3)
            fi, *en = self.pairs(d, on, self.eps[i][:, None] * self.eps[j][None], self.rad[i][:, None] + self.rad[j][None],
                                 q[i][:, None] * q[j][None])
            f[i] = fi
            total += torch.stack(en)
        return f, *total

    def gb_fixed(self):
        """Volumes and the covalent part of Gpol (Qiu et al.'s radii and constants)."""
        s, p = self.s, self.gb
        r = np.where(s.gbrad <= 0.01, 1.15, s.gbrad)
        vol = 4 * math.pi * r ** 3 / 3
        i = np.repeat(np.arange(s.n), np.diff(s.cov["off12"]))
        k, d = s.cov["idx12"], 1.01 * s.cov["d12"]
        h = r[i] * (1 + (r[k] ** 2 - r[i] ** 2 - d ** 2) / (2 * r[i] * d))
        np.subtract.at(vol, i, math.pi * h ** 2 * (3 * r[i] - h) / 3)
        vol = np.maximum(vol, 0.0)
        fixed = -166.0 / (r + p.DielectricOffset + p.P1)
        for c, o in (("12", p.P2), ("13", p.P3)):
            i = np.repeat(np.arange(s.n), np.diff(s.cov["off" + c]))
            np.add.at(fixed, i, o * vol[s.cov["idx" + c]] / s.cov["d" + c] ** 4)
        t = functools.partial(torch.tensor, dtype=torch.float64, device=self.dev)
        self.vol, self.fixed, self.gr = t(vol), t(fixed), t(s.gbrad)

    def still(self, x):
        """FastMode Generalized Born, vacuum Coulomb and LJ: x (b, n, 3)."""
        p, q = self.gb, self.q
        d = x[..., :, None, :] - x[..., None, :, :]
        eye = torch.eye(self.s.n, dtype=torch.bool, device=self.dev)
        r0 = torch.where(eye, 1.0, d.pow(2).sum(-1).sqrt())
        reach = self.on & (r0 * r0 <= p.GbsaStillCutoff ** 2)

        def gpol(r):
            u = r * r / (self.gr[:, None] + self.gr[None]) ** 2
            c = torch.where(u <= 1 / p.P5, (0.5 - 0.5 * torch.cos(u * p.P5 * math.pi)) ** 2, 1.0)
            return torch.where(reach, p.P4 * self.vol[None] * c / r ** 4, 0.0)
        a = -0.5 * ECONV / (self.fixed + gpol(r0).sum(-1)) + p.BornRadiusOffset
        r, a = r0.clone().requires_grad_(), a.requires_grad_()
        pre = -0.5 * ECONV * (1 / p.DielectricSolute - 1 / p.DielectricSolvent)
        within = ~eye & (r0 * r0 <= p.Cutoff ** 2)
        sw = self.switch(r, p.InnerCutoff, p.Cutoff)
        aa = a[..., :, None] * a[..., None, :]
        u = -r * r / (4 * aa)
        close = u > p.ExpApproxThreshold
        qq = q[:, None] * q[None]
        cross = torch.where(within & close, pre * qq / torch.sqrt(r * r + aa * torch.exp(u)) * sw, 0.0).sum((-1, -2))
        del u, aa
        s14, e14 = self.scaled14(p)
        ec = ECONV * (close.double() / p.DielectricSolute + (~close).double() / p.DielectricSolvent)
        elec = 0.5 * torch.where(within & self.on, ec * e14 * qq / r * sw, 0.0).sum((-1, -2))
        eps = s14 * self.eps[:, None] * self.eps[None]
        vdw = 0.5 * torch.where(within & self.on, self.lj(r, eps, self.rad[:, None] + self.rad[None], p.VdwInnerCutoff,
                                                          p.VdwCutoff), 0.0).sum((-1, -2))
        own = (pre * q * q / a).sum(-1)
        gr, ga = torch.autograd.grad((cross + elec + vdw + own).sum(), (r, a))
        weight = (a.detach() ** 2 / 166.0 * ga).detach()  # PD's factor for da/dGpol
        r1 = r0.clone().requires_grad_()
        gc, = torch.autograd.grad((weight * gpol(r1).sum(-1)).sum(), r1)
        g = (gr + gc) / r0
        g = g + g.transpose(-1, -2)
        return -(g[..., None] * d).sum(-2), [v.detach() for v in (cross + own, vdw, elec)]

    def surface(self, x):
        """LCPO forces and energy, one conformer (2-D products)."""
        x = x[self.heavy].detach().requires_grad_()
        d = (x[:, None] - x[None]).pow(2).sum(-1)
        n = len(x)
        m = (d.detach() < (self.lr[:, None] + self.lr[None]) ** 2) & ~torch.eye(n, dtype=torch.bool, device=self.dev)
        if int(m.sum(1).max()) > 80:  # PD keeps 80 neighbours: not what this formula says
            return None
        d = torch.where(m, d, 1.0).sqrt()
        r = self.lr[:, None]
        a = torch.where(m, 2 * math.pi * r * (r - d / 2 - (r * r - self.lr[None] ** 2) / (2 * d)), 0.0)
        mf = m.double()
        p1, p2, p3, p4 = self.lp.T
        area = p1 * 4 * math.pi * self.lr ** 2 + p2 * a.sum(1) + p3 * ((mf @ a) * mf).sum(1) + p4 * ((a @ a) * mf).sum(1)
        g, = torch.autograd.grad(ASP * area.sum(), x)
        buried = area.detach() < 0
        f = torch.zeros(self.s.n, 3, dtype=torch.float64, device=self.dev)
        f[self.heavy] = -torch.where(buried[:, None], 0.0, g)
        return f, ASP * torch.where(buried, 0.0, area.detach()).sum()

    def forces(self, x, sasa=None):
        """Forces and the energies (epot, vdw, elec, pol, surf, bond, angle, torsion, virial); `sasa` holds LCPO's stored part."""
        fb, eb, vir = self.bonded(x)
        x = x.to(self.dev)
        zero = torch.zeros_like(eb[0])
        if self.nb:
            f, vdw, elec, w = self.nonbonded(x)
            pol, vir = zero, w + (vir.to(self.dev) if vir is not None else zero)
        else:
            f, (pol, vdw, elec) = self.still(x)
            vir = zero
        f, surf = f + fb, zero
        if sasa is not None:
            f, surf = f + sasa[0], sasa[1]
        out = [vdw, elec, pol, surf, *eb]
        return f.cpu(), [v.cpu() for v in (sum(out), *out, vir)]


def philox(c, key):
    """Philox4x32-10 (Salmon et al. 2011): counters c (4 uint64 arrays of 32-bit values)."""
    k0, k1 = np.uint64(key & 0xFFFFFFFF), np.uint64(key >> 32)
    low = np.uint64(0xFFFFFFFF)
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ k0, p1 & low, (p0 >> np.uint64(32)) ^ c[3] ^ k1, p0 & low]
        k0, k1 = (k0 + np.uint64(0x9E3779B9)) & low, (k1 + np.uint64(0xBB67AE85)) & low
    return c


def normals(n, step, stream, seed):
    """Six unit normals per atom and step (Box-Muller)."""
    z = np.empty((n, 6))
    for k in range(3):
        c = philox([np.arange(n, dtype=np.uint64), *(np.full(n, v, dtype=np.uint64) for v in (step, stream, k))], seed)
        u1, u2 = ((((c[i] >> np.uint64(5)) << np.uint64(26)) | (c[i + 1] >> np.uint64(6))).astype(np.float64) + 1
                  for i in (0, 2))
        u1, u2 = u1 / 2.0 ** 53, u2 / 2.0 ** 53
        ln = np.sqrt(-2 * np.log(u1))
        z[:, 2 * k], z[:, 2 * k + 1] = ln * np.cos(-2 * math.pi * u2), ln * np.sin(-2 * math.pi * u2)
    return z


def langevin(g):
    """PD's c0, c1, c2, varr, varv, crv (series in g = friction * timestep, g <= 0.05)."""
    def series(first, *rest):
        return sum(c * g ** k for k, c in enumerate(rest, first))
    c0 = series(0, 1, -1, 1 / 2, -1 / 6, 1 / 24, -1 / 120)
    c1 = series(0, 1, -1 / 2, 1 / 6, -1 / 24, 1 / 120)
    c2 = series(0, 1 / 2, -1 / 6, 1 / 24, -1 / 120)
    varr = series(3, 2 / 3, -1 / 2, 7 / 30, -1 / 12, 31 / 1260)
    varv = series(1, 2, -2, 4 / 3, -2 / 3, 4 / 15)
    return c0, c1, c2, varr, varv, math.sqrt(3) * series(0, 1 / 2, -3 / 16, -17 / 1280, 17 / 6144)


def into_box(s, x):
    """cleanSpace: each molecule's centre brought into the box (three atoms per molecule)."""
    c = x.reshape(-1, 3, 3).mean(1)
    b = torch.tensor(s.box)
    return x + (-b * torch.ceil(c / b - 0.5)).repeat_interleave(3, 0)


def trajectory(case, seed, ref, x, v, temp, streams):
    """MD of one system, or of the conformers x (b, n, 3) of one: per-step energies (J), positions, velocities."""
    kind, dt = case["kind"], case["fs"] * 1e-15
    integ = case.get("integrator", "langevin")
    m = torch.tensor(ref.s.mass)[:, None]
    key = seed % 1000003
    co = langevin(FRICTION * dt)
    old, sasa, epot, ekin = torch.zeros_like(x), None, [], []
    for step in range(case["steps"]):
        if kind == "water" and step % UPDATE == 0:
            x = into_box(ref.s, x)
        if kind in ("gb", "batch") and step % SASA_EVERY == 0:
            if kind == "gb":
                sasa = ref.surface(x.to(ref.dev))
            else:
                each = [ref.surface(y) for y in x.to(ref.dev)]
                sasa = None if None in each else (torch.stack([f for f, _ in each]), torch.stack([e for _, e in each]))
            if sasa is None:
                return None
        f, en = ref.forces(x, sasa)
        f = f * JM
        epot.append(en[0] * KCAL)
        if integ == "langevin":
            c0, c1, c2, varr, varv, crv = co
            g = FRICTION * dt
            if step > 0:
                v = v + (1 - c0 / c1) * f * (dt / m) / g
        elif integ == "verlet":
            v = v + f * (0.5 * dt / m)
        elif step > 0:
            v = v + 2 * f * (dt / (6 * m))
        ekin.append((0.5 * m * v * v).sum((-1, -2)))
        if case.get("thermostat"):
            target = 1.5 * ref.s.n * KB * TEMP
            v = v * torch.sqrt(1 + dt * (target / ekin[-1] - 1) / TAU)
        if integ == "langevin":
            z = torch.tensor(np.stack([normals(ref.s.n, step, k, key) for k in streams]))
            z = z if x.dim() == 3 else z[0]
            n1, n2 = z[..., [0, 4, 3]], z[..., [2, 1, 5]]
            kt = KB * temp / m
            dv = torch.sqrt(kt * varv) * (crv * n1 + math.sqrt(1 - crv * crv) * n2)
            x = x + (dt * (c1 * v + c2 * f * (dt / m)) + torch.sqrt(kt * varr) / FRICTION * n1) / ANG
            v = c0 * v + c0 * c2 * f * (dt / m) / c1 + dv
        elif integ == "verlet":
            half = f * (0.5 * dt / m)
            x = x + dt * (v + 2 * half) / ANG
            v = v + 2 * half
        else:
            x = x + dt * (v + (4 * f - old) * (dt / (6 * m))) / ANG
            v = v + (5 * f - old) * (dt / (6 * m))
            old = f
    return torch.stack(epot), torch.stack(ekin), x, v


def exact(case, seed):
    kind, given = case["kind"], inputs(case, seed)
    if kind == "list":
        return None
    if kind == "batch":
        out = [None] * len(given)
        for s in {id(g[0]): g[0] for g in given}.values():
            mine = [k for k, g in enumerate(given) if g[0] is s]
            ref = Reference(s, gb=gb_kw(case), lcpo=True)
            for at in range(0, len(mine), 16):
                part = mine[at:at + 16]
                x, v = (torch.tensor(np.stack([given[k][c] for k in part])) for c in (1, 2))
                temp = torch.tensor([given[k][3] for k in part], dtype=torch.float64)[:, None, None]
                got = trajectory(case, seed, ref, x, v, temp, part)
                if got is None:
                    return None
                for b, k in enumerate(part):
                    out[k] = got[0][:, b], got[1][:, b], got[2][b]
        return dict(epot=torch.stack([o[0] for o in out], 1), ekin=torch.stack([o[1] for o in out], 1),
                    pos=torch.cat([o[2] for o in out]))
    s, x, v, _ = given[0]
    ref = Reference(s, **(dict(gb=gb_kw(case), lcpo=True) if kind == "gb" else dict(nb=nb_kw(case))))
    if kind == "mc":
        rows = []
        for y in moved(case, seed, x):
            _, vdw, elec, _ = ref.nonbonded(into_box(s, torch.tensor(y)).to(ref.dev))
            rows.append(torch.stack([vdw + elec, vdw, elec]).cpu() * KCAL)
        return dict(energies=torch.stack(rows))
    if kind == "point":
        f, en = ref.forces(into_box(s, torch.tensor(x)))
        epot, vdw, elec, _, _, bond, angle, tors, vir = (float(e) * KCAL for e in en)
        return dict(forces=f * JM, energies=torch.tensor([epot, vdw, elec, 0, 0, 0, bond, angle, tors, 0, vir, 0],
                                                         dtype=torch.float64))
    got = trajectory(case, seed, ref, torch.tensor(x), torch.tensor(v), TEMP, [0])
    return None if got is None else dict(zip(("epot", "ekin", "pos", "vel"), got))
