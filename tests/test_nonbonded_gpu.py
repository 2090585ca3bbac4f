"""GPU parity of the neighbour list and FF_NonBonded against the FP64 oracle.

Bars: pair set bit-exact (entries, bond orders, images, per-atom order);
cleanSpace positions bit-exact; total energy within 1e-5 relative; RMS force
error at most 1e-5 of the RMS force; forces bitwise reproducible run to run.
"""
import numpy as np
import pytest

from pd_amd import engine as G
from pd_amd import systems as S
from tests.helpers import O, energy_close, oracle_list, oracle_nb, rel_rms

pytestmark = pytest.mark.gpu

WATER_NB = dict(Cutoff=10.0, InnerCutoff=8.0, VdwCutoff=10.0, VdwInnerCutoff=8.0, ForceSwitch=1)


def _engine(s, nb_kw, padding, shadow=False):
    return G.engine_for(s, G.nb_params(**nb_kw), padding=padding, calc_shadow=shadow)


@pytest.mark.parametrize("n_waters,shadow", [(343, False), (512, False), (729, True), (1000, False)])
def test_water_pair_set_exact(n_waters, shadow):
    # 343 waters: a 21.7 A box, so Cutoff+Padding = 12 A exceeds half the box and
    # every pair takes PD's minimum-image loops; the larger boxes are decided
    # from the wrapped positions except near the limit.
    s = S.water_box(n_waters, seed=n_waters)
    print(f"case water n={n_waters} shadow={shadow}", flush=True)
    pos, counts, packed, _, _ = oracle_nb(s, WATER_NB, padding=2.0, shadow=shadow)
    e = _engine(s, WATER_NB, 2.0, shadow)
    e.build_list()
    assert e.full_update_count() == 1
    gpos = e.get_positions()
    assert np.array_equal(gpos, pos), "cleanSpace positions differ"
    gc, gp = e.get_pairs()
    assert np.array_equal(gc, counts)
    assert np.array_equal(gp, packed)


def _band_pairs(rlist):
    """A 512-water box (25 A) with positions on a 2^-20 A grid, and waters moved
    so that chosen O-O pairs lie at rlist exactly or 2^-34 / 2^-40 A inside or
    outside it, along x, directly and across the box face.  Every coordinate
    stays exact in FP64, so PD's r^2 lands on the limit or one side of it."""
    s = S.water_box(512, seed=77, box_len=25.0)
    s.pos = np.round(s.pos * 2.0**20) / 2.0**20
    L = s.box[0]
    deltas = [(0.0, True), (-2.0**-34, True), (2.0**-34, False), (-2.0**-40, True), (2.0**-40, False)]
    used, cases = set(), []
    ox = s.pos[0::3, 0]
    for cross in (False, True):
        lo, hi = ((-11.0, -1.0) if not cross else (2.0, 11.0))
        for d, expect in deltas:
            a = next(w for w in range(len(ox)) if lo <= ox[w] <= hi and w not in used)
            used.add(a)
            b = next(w for w in range(len(ox)) if w not in used)
            used.add(b)
            ia, ib = 3 * a, 3 * b
            target = s.pos[ia].copy()
            target[0] += rlist + d - (L if cross else 0.0)
            s.pos[ib:ib + 3] += target - s.pos[ib]
            assert s.pos[ib, 0] - s.pos[ia, 0] == rlist + d - (L if cross else 0.0)
            cases.append((ia, ib, expect))
    return s, cases


def _listed(counts, packed, a, b):
    start = np.concatenate([[0], np.cumsum(counts)])
    hi, lo = max(a, b), min(a, b)
    return lo in (packed[start[hi]:start[hi + 1]] & 0xFFFFFF)


def test_water_pair_set_exact_at_the_limit():
    s, cases = _band_pairs(12.0)
    print("case water band pairs", flush=True)
    pos, counts, packed, _, _ = oracle_nb(s, WATER_NB, padding=2.0)
    for a, b, expect in cases:  # the construction really puts pairs on both sides of the limit
        assert _listed(counts, packed, a, b) == expect, (a, b)
    e = _engine(s, WATER_NB, 2.0)
    e.build_list()
    gc, gp = e.get_pairs()
    assert np.array_equal(gc, counts)
    assert np.array_equal(gp, packed)


@pytest.mark.parametrize("n_waters,shadow", [(1, False), (1, True), (43, True), (2732, False)])
def test_pair_set_row_lengths(n_waters, shadow):
    # every pair is within the cutoff, so the rows have every length from none up
    # to 8,195 words: past one sort's 256 threads, each power of two, the longest
    # row sorted on the device (8,192), and many pieces of the transfer
    s = S.water_box(n_waters, seed=n_waters)
    s.box = None
    print(f"case rows n={3 * n_waters} shadow={shadow}", flush=True)
    counts, packed = oracle_list(s, O.clean_space(s), 80.0, 2.0, shadow)
    assert counts.max() == 3 * n_waters - 1
    e = G.engine_for(s, G.nb_params(Cutoff=80.0, InnerCutoff=70.0, VdwCutoff=80.0, VdwInnerCutoff=70.0),
                     padding=2.0, calc_shadow=shadow)
    e.build_list()
    gc, gp = e.get_pairs()
    assert np.array_equal(gc, counts)
    assert np.array_equal(gp, packed)


def test_peptide_vacuum_pair_set_exact():
    s = S.peptide_chain(20, seed=11)
    kw = dict(Cutoff=12.0, InnerCutoff=10.0, VdwCutoff=12.0, VdwInnerCutoff=10.0, ForceSwitch=0,
              EnergySwitch=1)
    print("case peptide20 vacuum", flush=True)
    pos, counts, packed, _, _ = oracle_nb(s, kw, padding=0.5)
    e = _engine(s, kw, 0.5)
    e.build_list()
    gc, gp = e.get_pairs()
    assert np.array_equal(gc, counts)
    assert np.array_equal(gp, packed)


@pytest.mark.parametrize("mode", ["force", "energy", "plain", "vdw_only", "elec_only", "vdwcor"])
def test_water_forces(mode):
    kw = dict(WATER_NB)
    if mode == "vdwcor":  # the long-range LJ correction (nonbonded.cpp:862-874)
        kw.update(VdwCor=1, VdwCorDensity=0.0334, VdwCorEpsilon=0.1521, VdwCorRadius=3.5364, VdwCorCutoff=10.0)
    if mode == "energy":
        kw.update(ForceSwitch=0, EnergySwitch=1)
    elif mode == "plain":
        kw.update(ForceSwitch=0, EnergySwitch=0)
    elif mode == "vdw_only":
        kw.update(DoElec=0)
    elif mode == "elec_only":
        kw.update(DoVdw=0)
    s = S.water_box(1000, seed=5)
    print(f"case water1000 mode={mode}", flush=True)
    pos, counts, packed, f_ref, e_ref = oracle_nb(s, kw, padding=2.0)
    e = _engine(s, kw, 2.0)
    e.build_list()
    f, en = e.compute(G.PDGPU_NONBONDED)
    err = rel_rms(f, f_ref)
    print(f"  rms force rel err {err:.2e}; epot {en['epot']:.6e} ref {e_ref['epot']:.6e}")
    assert err <= 1e-5
    for k in ("epot", "epot_vdw", "epot_elec"):
        ref = e_ref[k] if k != "epot" else e_ref["epot_vdw"] + e_ref["epot_elec"]
        assert energy_close(en[k], ref, e_ref["abs_sum"]), (k, en[k], ref, e_ref["abs_sum"])
    assert abs(en["virial"] - e_ref["virial"]) <= 1e-5 * abs(e_ref["virial"])


@pytest.mark.parametrize("n_waters", [1, 729, 2197, 6859])
def test_water_forces_by_size(n_waters):
    # one partly filled cluster, then boxes on each side of the lines between four, two
    # and one workgroup per group (the first two in FP64, two waves to a cluster).  A step's recorded energy is
    # summed by a workgroup of the next step's kernel, from the same partials.
    s = S.water_box(n_waters, seed=n_waters)
    if n_waters == 1:
        s.box = None
    print(f"case water n={n_waters} forces", flush=True)
    pos, counts, packed, f_ref, e_ref = oracle_nb(s, WATER_NB, padding=2.0)
    e = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0)
    e.build_list()
    f, en = e.compute(G.PDGPU_NONBONDED)
    f2, en2 = e.compute(G.PDGPU_NONBONDED)
    assert np.array_equal(f, f2) and en == en2
    assert np.array_equal(f, f_ref) if n_waters == 1 else rel_rms(f, f_ref) <= 1e-5
    assert energy_close(en["epot"], e_ref["epot_vdw"] + e_ref["epot_elec"], e_ref["abs_sum"])
    e.set_velocities(np.zeros((e.n, 3)))
    md = G.MDParams(integrator=G.PDGPU_VELOCITY_VERLET, components=G.PDGPU_NONBONDED, timestep=1e-15,
                    update_nlist=0, step_offset=0, total_steps=10, seed=1)
    trace = e.md(md, 2)[0]
    assert abs(trace[0] - en["epot"]) <= 1e-12 * e_ref["abs_sum"]


@pytest.mark.parametrize("cuts", [(10.0, 8.0, 8.0, 6.0), (8.0, 6.0, 10.0, 8.0)])
def test_water_forces_distinct_cutoffs(cuts):
    # VdwCutoff independent of Cutoff (nonbonded.cpp:722, 742): the kernel then
    # tests both cutoffs per pair instead of one
    c, ci, v, vi = cuts
    kw = dict(WATER_NB, Cutoff=c, InnerCutoff=ci, VdwCutoff=v, VdwInnerCutoff=vi)
    s = S.water_box(1000, seed=15)
    print(f"case water1000 cutoffs={cuts}", flush=True)
    pos, counts, packed, f_ref, e_ref = oracle_nb(s, kw, padding=2.0)
    e = _engine(s, kw, 2.0)
    e.build_list()
    gc, gp = e.get_pairs()
    assert np.array_equal(gc, counts) and np.array_equal(gp, packed)
    f, en = e.compute(G.PDGPU_NONBONDED)
    err = rel_rms(f, f_ref)
    print(f"  rms force rel err {err:.2e}")
    assert err <= 1e-5
    for k in ("epot", "epot_vdw", "epot_elec"):
        ref = e_ref[k] if k != "epot" else e_ref["epot_vdw"] + e_ref["epot_elec"]
        assert energy_close(en[k], ref, e_ref["abs_sum"]), (k, en[k], ref, e_ref["abs_sum"])


def test_peptide_vacuum_forces_with_14():
    s = S.peptide_chain(20, seed=3)
    kw = dict(Cutoff=12.0, InnerCutoff=10.0, VdwCutoff=12.0, VdwInnerCutoff=10.0, ForceSwitch=0,
              EnergySwitch=1, Vdw14Scaling=0.5, Elec14Scaling=0.83333)
    print("case peptide20 forces", flush=True)
    pos, counts, packed, f_ref, e_ref = oracle_nb(s, kw, padding=0.5)
    e = _engine(s, kw, 0.5)
    e.build_list()
    f, en = e.compute(G.PDGPU_NONBONDED)
    assert rel_rms(f, f_ref) <= 1e-5
    ref = e_ref["epot_vdw"] + e_ref["epot_elec"]
    assert abs(en["epot"] - ref) <= 1e-5 * abs(ref)


def test_energy_only_matches_oracle():
    """FF_NonBonded::calcEnergies_Full (nonbonded.cpp:1184-1202), the MC energy
    path, against the oracle's energies at the same positions: the energy-only
    kernel, not the force kernel, is what is compared."""
    for mode, kw in (("force", WATER_NB), ("energy", dict(WATER_NB, ForceSwitch=0, EnergySwitch=1))):
        s = S.water_box(729, seed=31)
        print(f"case energy-only water729 {mode}", flush=True)
        pos, counts, packed, f_ref, e_ref = oracle_nb(s, kw, padding=2.0)
        e = _engine(s, kw, 2.0)
        e.build_list()
        _, en = e.compute(G.PDGPU_NONBONDED | G.PDGPU_ENERGY_ONLY, forces=False)
        for k in ("epot", "epot_vdw", "epot_elec"):
            ref = e_ref[k] if k != "epot" else e_ref["epot_vdw"] + e_ref["epot_elec"]
            assert energy_close(en[k], ref, e_ref["abs_sum"]), (mode, k, en[k], ref)
        assert abs(en["virial"] - e_ref["virial"]) <= 1e-5 * abs(e_ref["virial"])
    s = S.peptide_chain(20, seed=3)
    kw = dict(Cutoff=12.0, InnerCutoff=10.0, VdwCutoff=12.0, VdwInnerCutoff=10.0, ForceSwitch=0,
              EnergySwitch=1, Vdw14Scaling=0.5, Elec14Scaling=0.83333)
    pos, counts, packed, f_ref, e_ref = oracle_nb(s, kw, padding=0.5)
    e = _engine(s, kw, 0.5)
    e.build_list()
    _, en = e.compute(G.PDGPU_NONBONDED | G.PDGPU_ENERGY_ONLY, forces=False)
    ref = e_ref["epot_vdw"] + e_ref["epot_elec"]
    assert abs(en["epot"] - ref) <= 1e-5 * abs(ref)


def test_forces_bitwise_reproducible():
    s = S.water_box(1000, seed=9)
    e = _engine(s, WATER_NB, 2.0)
    e.build_list()
    f1, e1 = e.compute(G.PDGPU_NONBONDED)
    f2, e2 = e.compute(G.PDGPU_NONBONDED)
    e.build_list()
    f3, e3 = e.compute(G.PDGPU_NONBONDED)
    assert np.array_equal(f1, f2) and np.array_equal(f1, f3)
    assert e1 == e2 == e3


def test_newton_third_law_fixed_point():
    s = S.water_box(512, seed=2)
    e = _engine(s, WATER_NB, 2.0)
    e.build_list()
    f, _ = e.compute(G.PDGPU_NONBONDED)
    # fixed-point sums cancel exactly; the J/m conversion leaves only rounding
    # each pair's two halves are rounded to fixed point in different partial
    # sums, so the net force is zero to FP32 rounding, not exactly
    assert np.abs(f.sum(axis=0)).max() <= 1e-5 * np.abs(f).max()


def test_setup_rejects_cutoff_beyond_half_box():
    s = S.water_box(216, seed=1)  # 18.6 A box
    e = G.Engine(s.n)
    e.set_atom_params(s.radius, s.epsilon, s.charge, s.mass)
    e.set_space(s.box)
    with pytest.raises(G.PdGpuError) as ex:
        e.setup_nonbonded(G.nb_params(**WATER_NB))
    assert ex.value.code == -3


def test_relaxed_water_energy_relative():
    """A box relaxed by device Langevin dynamics has a well-conditioned total
    energy; there the 1e-5 relative bar applies without the summation allowance."""
    import tests.test_md_gpu as M
    s = S.water_box(1000, seed=21)
    e = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0, bonded=True)
    md = G.MDParams(integrator=G.PDGPU_LANGEVIN, components=G.PDGPU_NONBONDED | G.PDGPU_BONDED,
                    timestep=0.5e-15, temperature=300.0, fric_coeff=5e13, update_nlist=10,
                    step_offset=0, total_steps=100000, seed=7)
    e.md(md, 400)
    s2 = s.copy()
    s2.pos = e.get_positions()
    pos, counts, packed, f_ref, e_ref = oracle_nb(s2, WATER_NB, padding=2.0)
    e2 = _engine(s2, WATER_NB, 2.0)
    e2.build_list()
    f, en = e2.compute(G.PDGPU_NONBONDED)
    ref = e_ref["epot_vdw"] + e_ref["epot_elec"]
    print(f"relaxed: E={ref * 6.0221418e23 / 4184:.3f} kcal/mol rel err {abs(en['epot'] - ref) / abs(ref):.2e} "
          f"force rms rel {rel_rms(f, f_ref):.2e}")
    assert abs(en["epot"] - ref) <= 1e-5 * abs(ref)
    assert rel_rms(f, f_ref) <= 1e-5
