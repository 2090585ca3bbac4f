"""GPU parity of FF_GeneralizedBorn_Still (FastMode) against the FP64 oracle.

Bars: Born radii within 1e-6 relative; each energy term within 1e-5 relative
(plus the FP32 summation allowance for cancelling sums); RMS force error at
most 1e-5 of the RMS force; forces bitwise reproducible.
"""
import numpy as np
import pytest

from oracle import oracle as O
from pd_amd import engine as G
from pd_amd import systems as S
from tests.helpers import rel_rms

pytestmark = pytest.mark.gpu

ALL_PAIRS = dict(Cutoff=999.0, InnerCutoff=999.0, VdwCutoff=999.0, VdwInnerCutoff=999.0, GbsaStillCutoff=999.0,
                 DielectricSolvent=78.5, Vdw14Scaling=0.5, Elec14Scaling=0.83333)
SWITCHED = dict(Cutoff=12.0, InnerCutoff=10.0, VdwCutoff=12.0, VdwInnerCutoff=10.0, GbsaStillCutoff=10.0,
                DielectricSolvent=80.0, Vdw14Scaling=0.5, Elec14Scaling=0.83333)


def oracle_gb(s, kw):
    p = O.gb_params(**kw)
    bo = O.bond_order(s)
    cut = max(p.Cutoff, p.VdwCutoff)
    counts, packed = O.build_list(s, s.pos, cut, 0.5, True, bo)
    Vj, t123, _ = O.gb_fixed_terms(s, p)
    born = O.gb_radii(s, s.pos, Vj, t123, p, counts, packed)
    f, e = O.gb_forces_fast(s, s.pos, Vj, born, p, counts, packed)
    return born, f, e


def gpu_gb(s, kw):
    e = G.engine_for(s, None)
    e.setup_gb(G.gb_params(**kw), s.gbrad, s.cov)
    f, en = e.compute(G.PDGPU_GB)
    return e, f, en


# 1 residue (22 atoms): one partly filled 64-atom tile; 4 residues (73 atoms):
# a full tile and a partly filled one
@pytest.mark.parametrize("n_res,seed,kw", [(20, 1, ALL_PAIRS), (20, 2, SWITCHED), (60, 3, ALL_PAIRS),
                                           (60, 4, SWITCHED), (1, 5, ALL_PAIRS), (4, 6, SWITCHED)],
                         ids=["ala20-all", "pep20-switch", "pep60-all", "pep60-switch", "pep1-all",
                              "pep4-switch"])
def test_gb_forces_energies(n_res, seed, kw):
    s = S.peptide_chain(n_res, seed=seed)
    print(f"case peptide{n_res} seed={seed} {kw['Cutoff']}", flush=True)
    born_ref, f_ref, e_ref = oracle_gb(s, kw)
    e, f, en = gpu_gb(s, kw)
    born = e.born_radii()
    rb = np.abs(born - born_ref).max() / np.abs(born_ref).max()
    ferr = rel_rms(f, f_ref)
    print(f"  born max rel {rb:.2e}  force rms rel {ferr:.2e}")
    for k in ("epot", "epot_pol", "epot_pol_self", "epot_pol_cross", "epot_vdw", "epot_elec"):
        print(f"  {k:15s} gpu {en[k]:.9e} ref {e_ref[k]:.9e} rel {abs(en[k] - e_ref[k]) / abs(e_ref[k]):.2e}")
    assert rb <= 1e-6
    assert ferr <= 1e-5
    scale = coulomb_abs_sum(s, kw)
    for k in ("epot", "epot_pol", "epot_pol_self", "epot_pol_cross", "epot_vdw", "epot_elec"):
        allowance = 1e-6 * scale if k in ("epot_elec", "epot") else 0.0
        assert abs(en[k] - e_ref[k]) <= 1e-5 * abs(e_ref[k]) + allowance, k


def coulomb_abs_sum(s, kw):
    """sum over non-bonded/1-4 pairs within Cutoff of |econv q_i q_j / r| (J): the
    condition scale of the vacuum Coulomb total, for the FP32 summation allowance."""
    from pd_amd import units as U
    bo = O.bond_order(s)
    counts, packed = O.build_list(s, s.pos, kw["Cutoff"], 0.0, False, bo)
    i = np.repeat(np.arange(s.n), counts)
    j = (packed & 0xFFFFFF).astype(np.int64)
    order = (packed >> 24) & 7
    r = np.linalg.norm(s.pos[i] - s.pos[j], axis=1)
    keep = order >= 3
    return float(np.sum(np.abs(U.ECONV_JOULE * s.charge[i] * s.charge[j] / r)[keep]))


def test_gb_far_pairs_use_solvent_dielectric():
    """Pairs with uGB <= ExpApproxThreshold drop the GB cross term and use eps_solvent
    for Coulomb (gbff.cpp:1659-1678): exercised by a spread-out chain."""
    s = S.peptide_chain(40, seed=9, phi_mu=-120.0, psi_mu=130.0)
    born_ref, f_ref, e_ref = oracle_gb(s, ALL_PAIRS)
    e, f, en = gpu_gb(s, ALL_PAIRS)
    assert rel_rms(f, f_ref) <= 1e-5
    assert abs(en["epot"] - e_ref["epot"]) <= 1e-5 * abs(e_ref["epot"])


def test_gb_and_lcpo_reject_a_periodic_space():
    """PD's GB and LCPO take raw displacements (gbff.cpp:459, lcpo.cpp:477), so
    they have no meaning in a periodic box: the engine refuses them there."""
    s = S.peptide_chain(4, seed=2)
    e = G.engine_for(s, None)
    e.setup_gb(G.gb_params(**ALL_PAIRS), s.gbrad, s.cov)
    use, rad, P = S.lcpo_params(s)
    e.setup_lcpo(G.LCPOParams(GlobalASP=0.009, UpdateSasa=5), rad, P, use)
    e.compute(G.PDGPU_GB | G.PDGPU_SASA)
    e.set_space(np.array([60.0, 60.0, 60.0]))
    for comp in (G.PDGPU_GB, G.PDGPU_SASA):
        with pytest.raises(G.PdGpuError, match="vacuum"):
            e.compute(comp)
    e.set_space(None)
    e.compute(G.PDGPU_GB | G.PDGPU_SASA)


def test_gb_reproducible():
    s = S.peptide_chain(30, seed=5)
    e, f1, e1 = gpu_gb(s, ALL_PAIRS)
    f2, e2 = e.compute(G.PDGPU_GB)
    assert np.array_equal(f1, f2) and e1 == e2


def oracle_gb_born(s, kw):
    p = O.gb_params(**kw)
    bo = O.bond_order(s)
    counts, packed = O.build_list(s, s.pos, max(p.Cutoff, p.VdwCutoff), 0.5, True, bo)
    Vj, t123, _ = O.gb_fixed_terms(s, p)
    born = O.gb_radii(s, s.pos, Vj, t123, p, counts, packed)
    f, e, pol = O.gb_forces_born(s, s.pos, Vj, born, p, counts, packed)
    return f, e, pol


@pytest.mark.parametrize("which,kw", [("amber-ala10", ALL_PAIRS), ("amber-rand40", ALL_PAIRS),
                                      ("amber-rand40", SWITCHED), ("spread40", ALL_PAIRS)])
def test_gb_non_fastmode_forces_energies(which, kw):
    """calcForces with FastMode off (FF_NonBonded::calcForces + calcBornForces,
    gbff.cpp:186-196, 1189-1437) against the oracle: forces, the total energy and
    its vdW / Coulomb terms; the ene.epot_pol* terms stay zero as in PD.  The
    spread-out chain has pairs beyond the exp threshold (1/r cross term)."""
    from pd_amd import forcefield as F
    if which == "amber-ala10":
        s = F.new_protein(["ALA"] * 10)
    elif which == "amber-rand40":
        s = F.random_peptide(40, 21)
    else:
        s = S.peptide_chain(40, seed=9, phi_mu=-120.0, psi_mu=130.0)
    if which != "spread40":
        kw = dict(kw, Vdw14Scaling=s.ff.vdw14, Elec14Scaling=s.ff.elec14)
    print(f"case non-fast {which} cutoff {kw['Cutoff']}", flush=True)
    f_ref, e_ref, pol = oracle_gb_born(s, kw)
    e = G.engine_for(s, None)
    e.setup_gb(G.gb_params(FastMode=0, **kw), s.gbrad, s.cov)
    f, en = e.compute(G.PDGPU_GB)
    ferr = rel_rms(f, f_ref)
    print(f"  force rms rel {ferr:.2e}; epot gpu {en['epot']:.9e} ref {e_ref['epot']:.9e}; "
          f"pol {pol[0]:.6e}")
    assert ferr <= 1e-5
    scale = coulomb_abs_sum(s, kw)
    for k in ("epot", "epot_vdw", "epot_elec"):
        allowance = 1e-6 * scale if k in ("epot_elec", "epot") else 0.0
        assert abs(en[k] - e_ref[k]) <= 1e-5 * abs(e_ref[k]) + allowance, k
    assert en["epot_pol"] == en["epot_pol_self"] == en["epot_pol_cross"] == 0.0
    # the same engine in FastMode differs (no 1/r tail, solvent Coulomb beyond the threshold)
    e2 = G.engine_for(s, None)
    e2.setup_gb(G.gb_params(**kw), s.gbrad, s.cov)
    f2, en2 = e2.compute(G.PDGPU_GB)
    assert en2["epot_pol"] != 0.0


def test_gb_split_variants_and_autotuner():
    """Every work split of the GB tile kernels (1, 2, 4 wavefronts per tile pair)
    meets the oracle bars and is bitwise reproducible; the autotuner's choice is
    one of them and gives what setting it by hand gives; a batch with a split
    equals its single-system engines with the same split."""
    from pd_amd import forcefield as F
    s = F.random_peptide(50, 8)
    kw = dict(ALL_PAIRS, Vdw14Scaling=s.ff.vdw14, Elec14Scaling=s.ff.elec14)
    born_ref, f_ref, e_ref = oracle_gb(s, kw)
    e = G.engine_for(s, None)
    e.setup_gb(G.gb_params(**kw), s.gbrad, s.cov)
    f1, en1 = e.compute(G.PDGPU_GB)
    for sp in ((2, 2, 2), (4, 4, 4), (1, 4, 2)):
        print(f"case split {sp}", flush=True)
        e.set_gb_split(sp)
        f, en = e.compute(G.PDGPU_GB)
        f2, en2 = e.compute(G.PDGPU_GB)
        assert np.array_equal(f, f2) and en == en2
        assert rel_rms(f, f_ref) <= 1e-5 and rel_rms(f, f1) <= 1e-6
        assert abs(en["epot"] - e_ref["epot"]) <= 1e-5 * abs(e_ref["epot"]) + 1e-6 * coulomb_abs_sum(s, kw)
    choice, us = e.autotune_gb()
    print(f"autotuner: split {choice.tolist()}, us {np.round(us, 2).tolist()}", flush=True)
    assert set(choice.tolist()) <= {1, 2, 4} and (us > 0).all()
    fa, ena = e.compute(G.PDGPU_GB)
    # the choice is kept for the process: an engine of the same shape starts with it
    e2 = G.engine_for(s, None)
    e2.setup_gb(G.gb_params(**kw), s.gbrad, s.cov)
    fb, enb = e2.compute(G.PDGPU_GB)
    assert np.array_equal(fa, fb) and ena == enb
    e2.set_gb_split(choice)
    fc, enc = e2.compute(G.PDGPU_GB)
    assert np.array_equal(fa, fc) and ena == enc
    # a batch of uneven chains at split (2, 4, 2) against its members at the same split
    chains = [F.random_peptide(n, 30 + n) for n in (5, 17, 33)]
    engines = []
    for c in chains:
        en_ = G.engine_for(c, None)
        en_.setup_gb(G.gb_params(**dict(ALL_PAIRS, Vdw14Scaling=c.ff.vdw14, Elec14Scaling=c.ff.elec14)), c.gbrad,
                     c.cov)
        en_.set_gb_split((2, 4, 2))
        engines.append(en_)
    b = G.Batch(engines)
    b.set_gb_split((2, 4, 2))
    fb_, eb_ = b.compute(G.PDGPU_GB)
    for k, en_ in enumerate(engines):
        f_, e_ = en_.compute(G.PDGPU_GB)
        assert np.array_equal(fb_[k], f_), k
    bc, bus = b.autotune_gb()
    assert set(bc.tolist()) <= {1, 2, 4}


@pytest.mark.parametrize("n_atoms", [63, 64, 65, 128, 129, 257, 640])
@pytest.mark.parametrize("kw", [ALL_PAIRS, SWITCHED], ids=["all", "switch"])
def test_gb_tile_edges_and_far_tiles(n_atoms, kw):
    """Systems cut at the edges of the 64-atom tiles, stretched so that distant tile
    pairs take the far loops (one i tile and two, and the single tile of an odd count),
    against the oracle at the bars above; every split gives the same bits."""
    s = S.peptide_chain(44, seed=31, phi_mu=-120.0, psi_mu=130.0)
    # the first n_atoms atoms, with the covalent partners among them
    def cut(off, idx, *more):
        keep = [k for i in range(n_atoms) for k in range(s.cov[off][i], s.cov[off][i + 1]) if s.cov[idx][k] < n_atoms]
        cnt = [sum(s.cov[idx][k] < n_atoms for k in range(s.cov[off][i], s.cov[off][i + 1])) for i in range(n_atoms)]
        return {off: np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32), idx: s.cov[idx][keep],
                **{m: s.cov[m][keep] for m in more}}
    assert s.n >= 640
    s.cov = {**cut("off12", "idx12", "d12"), **cut("off13", "idx13", "d13"), **cut("off14", "idx14")}
    for f in ("pos", "radius", "epsilon", "charge", "mass", "gbrad", "resid"):
        setattr(s, f, getattr(s, f)[:n_atoms].copy())
    s.mol_last = np.array([n_atoms - 1], dtype=np.int32)
    print(f"case tile edges n={n_atoms} cutoff {kw['Cutoff']}", flush=True)
    born_ref, f_ref, e_ref = oracle_gb(s, kw)
    e, f, en = gpu_gb(s, kw)
    assert np.abs(e.born_radii() - born_ref).max() <= 1e-6 * np.abs(born_ref).max()
    assert rel_rms(f, f_ref) <= 1e-5
    scale = coulomb_abs_sum(s, kw)
    for k in ("epot", "epot_pol", "epot_vdw", "epot_elec"):
        assert abs(en[k] - e_ref[k]) <= 1e-5 * abs(e_ref[k]) + 1e-6 * scale, k
    for sp in ((1, 1, 1), (2, 2, 2), (4, 4, 4)):
        e.set_gb_split(sp)
        assert np.array_equal(e.compute(G.PDGPU_GB)[0], f), sp


@pytest.mark.parametrize("kw", [ALL_PAIRS, SWITCHED], ids=["all", "switch"])
def test_gb_plain_comparator_matches_oracle(kw):
    """The plain FP64 comparator (one thread per atom, FP64 sums) against the
    oracle at FP64 bars: it is the baseline of the batched-engine speedup."""
    from pd_amd import forcefield as F
    s = F.random_peptide(30, 11)
    kw = dict(kw, Vdw14Scaling=s.ff.vdw14, Elec14Scaling=s.ff.elec14)
    print(f"case plain comparator cutoff {kw['Cutoff']}", flush=True)
    born_ref, f_ref, e_ref = oracle_gb(s, kw)
    e = G.engine_for(s, None)
    e.setup_gb(G.gb_params(**kw), s.gbrad, s.cov)
    e.set_gb_plain(True)
    f, en = e.compute(G.PDGPU_GB)
    born = e.born_radii()
    assert np.abs(born - born_ref).max() <= 1e-12 * np.abs(born_ref).max()
    assert rel_rms(f, f_ref) <= 1e-8
    for k in ("epot", "epot_pol", "epot_pol_self", "epot_pol_cross", "epot_vdw", "epot_elec"):
        assert en[k] == pytest.approx(e_ref[k], rel=1e-9), k


def test_gb_md_with_finite_cutoffs_matches_pd_list():
    """PD's GB takes its pairs from the neighbour list built at Cutoff + Padding at
    the last rebuild; the engine takes every pair within the cutoffs at the current
    positions.  After 25 Langevin steps with finite cutoffs (12/10 A, Still 10 A,
    padding 2 A, rebuilds at steps 0, 10, 20), the engine's forces and energies equal
    the oracle's computed over the list built at step 20's positions."""
    from pd_amd import forcefield as F
    s = F.random_peptide(30, 21)
    kw = dict(SWITCHED, Vdw14Scaling=s.ff.vdw14, Elec14Scaling=s.ff.elec14)
    e = G.engine_for(s, None, padding=2.0, bonded=True)
    e.setup_gb(G.gb_params(**kw), s.gbrad, s.cov)
    comps = G.PDGPU_GB | G.PDGPU_BONDED
    md = G.MDParams(integrator=G.PDGPU_LANGEVIN, components=comps, timestep=2e-15, temperature=300.0,
                    fric_coeff=5e12, update_nlist=10, step_offset=0, total_steps=1000, seed=3)
    e.md(md, 20)
    p20 = e.get_positions()
    md.step_offset = 20
    e.md(md, 5)
    p25 = e.get_positions()
    f, en = e.compute(G.PDGPU_GB)
    p = O.gb_params(**kw)
    bo = O.bond_order(s)
    counts, packed = O.build_list(s, p20, max(p.Cutoff, p.VdwCutoff), 2.0, True, bo)
    Vj, t123, _ = O.gb_fixed_terms(s, p)
    born = O.gb_radii(s, p25, Vj, t123, p, counts, packed)
    f_ref, e_ref = O.gb_forces_fast(s, p25, Vj, born, p, counts, packed)
    moved = np.abs(p25 - p20).max()
    print(f"largest move since the rebuild {moved:.3f} A; force rms rel {rel_rms(f, f_ref):.2e}", flush=True)
    assert moved < 1.0  # every pair's distance changed by less than the padding
    assert rel_rms(f, f_ref) <= 1e-5
    for k in ("epot", "epot_pol", "epot_vdw", "epot_elec"):
        assert abs(en[k] - e_ref[k]) <= 1e-5 * abs(e_ref[k]) + 1e-6 * coulomb_abs_sum(s, kw), k
