"""GPU parity of FF_Bonded and of the device-resident integrators against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from pd_amd import engine as G
from pd_amd import systems as S
from pd_amd import units as U
from tests.helpers import rel_rms

pytestmark = pytest.mark.gpu

WATER_NB = dict(Cutoff=10.0, InnerCutoff=8.0, VdwCutoff=10.0, VdwInnerCutoff=8.0, ForceSwitch=1)


def mb_velocities(s, temp, seed):
    rng = np.random.default_rng(seed)
    sig = np.sqrt(U.KB * temp / s.mass)
    return rng.normal(size=(s.n, 3)) * sig[:, None]


@pytest.mark.parametrize("which", ["water", "peptide"])
def test_bonded_forces(which):
    s = S.water_box(512, seed=4) if which == "water" else S.peptide_chain(30, seed=8)
    rng = np.random.default_rng(1)
    pos = s.pos + rng.normal(scale=0.05, size=s.pos.shape)
    f_ref, e_ref = O.bonded_forces(s, pos)
    e = G.engine_for(s, None, bonded=True)
    e.set_positions(pos)
    f, en = e.compute(G.PDGPU_BONDED)
    assert rel_rms(f, f_ref) <= 1e-9
    for k in ("epot_bond", "epot_angle", "epot_torsion"):
        assert abs(en[k] - e_ref[k]) <= 1e-10 * max(abs(e_ref[k]), 1e-30) + 1e-30, k


def test_velocity_verlet_step_bit_exact():
    s = S.water_box(512, seed=6)
    e = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0, bonded=True)
    e.build_list()
    v0 = mb_velocities(s, 300.0, 3)
    e.set_velocities(v0)
    comps = G.PDGPU_NONBONDED | G.PDGPU_BONDED
    f, _ = e.compute(comps)
    p0 = e.get_positions()
    md = G.MDParams(integrator=G.PDGPU_VELOCITY_VERLET, components=comps, timestep=1e-15,
                    update_nlist=10, step_offset=0, total_steps=1, seed=1)
    ep, ek = e.md(md, 1)
    pos = p0.copy(); vel = v0.copy()
    ke = O.vv_step(s.mass, 1e-15, f, pos, vel)
    assert np.array_equal(e.get_positions(), pos)
    assert np.array_equal(e.get_velocities(), vel)
    assert ek[0] == pytest.approx(ke, rel=1e-14)


def test_beeman_steps_bit_exact():
    """Three Beeman steps of a 3-step protocol (no kick on step 0, no move on the
    last) against the oracle fed the engine's own forces; the old forces start at
    zero and persist between calls."""
    s = S.water_box(512, seed=6)
    e = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0, bonded=True)
    e.build_list()
    v0 = mb_velocities(s, 300.0, 3)
    e.set_velocities(v0)
    comps = G.PDGPU_NONBONDED | G.PDGPU_BONDED
    pos = e.get_positions()
    vel = v0.copy()
    fold = np.zeros_like(pos)
    for st in range(3):
        print(f"case beeman step {st}", flush=True)
        f, _ = e.compute(comps)
        md = G.MDParams(integrator=G.PDGPU_BEEMAN, components=comps, timestep=1e-15,
                        update_nlist=10, step_offset=st, total_steps=3, seed=1)
        ep, ek = e.md(md, 1)
        ke = O.beeman_step(s.mass, 1e-15, st, 3, f, fold, pos, vel)
        assert np.array_equal(e.get_positions(), pos)
        assert np.array_equal(e.get_velocities(), vel)
        assert ek[0] == pytest.approx(ke, rel=1e-14)


def test_md_recovers_from_list_overflow_at_a_rebuild():
    """A rebuild inside pdgpu_md whose list outgrows the capacity sized at the first
    build (here from a 4x expanded chain) is redone with room before the step is
    integrated: the run equals one that started from the compact chain."""
    s = S.peptide_chain(20, seed=11)
    kw = dict(Cutoff=12.0, InnerCutoff=10.0, VdwCutoff=12.0, VdwInnerCutoff=10.0, ForceSwitch=0,
              EnergySwitch=1)
    comps = G.PDGPU_NONBONDED | G.PDGPU_BONDED
    sparse = s.copy()
    c = s.pos.mean(axis=0)
    sparse.pos = c + 4.0 * (s.pos - c)
    a = G.engine_for(sparse, G.nb_params(**kw), padding=0.5, bonded=True)
    a.build_list()
    a.set_positions(s.pos)
    b = G.engine_for(s, G.nb_params(**kw), padding=0.5, bonded=True)
    v0 = mb_velocities(s, 300.0, 5)
    a.set_velocities(v0)
    b.set_velocities(v0)
    md = G.MDParams(integrator=G.PDGPU_VELOCITY_VERLET, components=comps, timestep=1e-15, update_nlist=2,
                    step_offset=0, total_steps=5, seed=1)
    print("case overflow retry", flush=True)
    a.set_timing(True)
    b.set_timing(True)
    ea, ka = a.md(md, 5)
    eb, kb = b.md(md, 5)
    assert a.kernel_time("pair_search")[1] == b.kernel_time("pair_search")[1] + 1  # the retried build
    assert a.full_update_count() == b.full_update_count() + 1  # a's build before the run
    assert np.array_equal(a.get_positions(), b.get_positions())
    assert np.array_equal(ea, eb) and np.array_equal(ka, kb)


def _thermo_engine():
    s = S.water_box(512, seed=6)
    e = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0, bonded=True)
    e.build_list()
    v0 = mb_velocities(s, 300.0, 3)
    e.set_velocities(v0)
    return s, e, v0


@pytest.mark.parametrize("integ,thermo", [("vv", "berendsen"), ("vv", "andersen"), ("beeman", "berendsen"),
                                          ("beeman", "andersen")])
def test_thermostat_steps_match_oracle(integ, thermo):
    """Two steps (step 1 of each protocol kicks, thermostats, moves) with the
    momentum removal of run_core at step 1, against the oracle composed as PD's
    step: kick, kinetic energy, applyThermostat, move; then the momentum step."""
    s, e, v0 = _thermo_engine()
    comps = G.PDGPU_NONBONDED | G.PDGPU_BONDED
    I = G.PDGPU_VELOCITY_VERLET if integ == "vv" else G.PDGPU_BEEMAN
    T = G.PDGPU_BERENDSEN if thermo == "berendsen" else G.PDGPU_ANDERSEN
    rate = 0.3 * s.n ** (2.0 / 3.0)  # 30% of the atoms reassigned per step at 1 fs
    seed, stream, dt, tau = 0xABCDEF, 4, 1e-15, 50e-15
    pos = e.get_positions()
    vel = v0.copy()
    fold = np.zeros_like(pos)
    for st in range(2):
        print(f"case {integ} {thermo} step {st}", flush=True)
        f, _ = e.compute(comps)
        md = G.MDParams(integrator=I, components=comps, timestep=dt, temperature=280.0, update_nlist=10,
                        step_offset=st, total_steps=3, seed=seed, noise_stream=stream, thermostat=T,
                        remove_momentum=1, berendsen_tau=tau, andersen_rate=rate)
        ep, ek = e.md(md, 1)
        if integ == "vv":
            O.vv_kick(s.mass, dt, f, vel)
        else:
            O.beeman_kick(s.mass, dt, st, f, vel)
        K = O.kinetic_energy(s.mass, vel)
        if thermo == "berendsen":
            O.berendsen(K, 280.0, dt, tau, vel)
        else:
            assert O.andersen(s.mass, 280.0, rate, dt, seed, stream, st, vel) > 0
        if integ == "vv":
            O.vv_move(s.mass, dt, f, pos, vel)
        else:
            O.beeman_move(s.mass, dt, st, 3, f, fold, pos, vel)
        if st > 0:
            O.zero_momentum(s.mass, pos, vel)
        assert ek[0] == pytest.approx(K, rel=1e-13)
        np.testing.assert_allclose(e.get_positions(), pos, rtol=0, atol=1e-12)
        np.testing.assert_allclose(e.get_velocities(), vel, rtol=1e-11, atol=1e-11 * np.abs(vel).max())


def test_langevin_step_matches_oracle():
    s = S.peptide_chain(10, seed=2)
    e = G.engine_for(s, None, bonded=True)
    v0 = mb_velocities(s, 300.0, 4)
    e.set_velocities(v0)
    f, _ = e.compute(G.PDGPU_BONDED)
    p0 = e.get_positions()
    seed = 0x1234_5678_9ABC
    md = G.MDParams(integrator=G.PDGPU_LANGEVIN, components=G.PDGPU_BONDED, timestep=2e-15,
                    temperature=300.0, fric_coeff=1e12, update_nlist=0, step_offset=3, total_steps=10,
                    seed=seed)
    e.md(md, 1)
    noise = np.array([O.langevin_noise(seed, 0, 3, i) for i in range(s.n)])
    pos = p0.copy(); vel = v0.copy()
    O.langevin_step(s.mass, 2e-15, 1e12, 300.0, 3, 10, f, noise, pos, vel)
    np.testing.assert_allclose(e.get_positions(), pos, rtol=0, atol=1e-12)
    np.testing.assert_allclose(e.get_velocities(), vel, rtol=1e-9, atol=1e-9 * np.abs(vel).max())


@pytest.mark.parametrize("integ", ["vv", "beeman", "langevin"])
def test_berendsen_barostat_steps_match_oracle(integ):
    """Two steps with the Berendsen barostat: the device's pressure, scaling
    factor, positions, velocities and box against the oracle composed as PD's
    step (kick, calcKineticEnergy with the pressure, applyBarostat, move), fed
    the engine's own forces and virial."""
    s, e, v0 = _thermo_engine()
    comps = G.PDGPU_NONBONDED | G.PDGPU_BONDED
    I = {"vv": G.PDGPU_VELOCITY_VERLET, "beeman": G.PDGPU_BEEMAN, "langevin": G.PDGPU_LANGEVIN}[integ]
    dt, seed, gamma = 1e-15, 0x5EED, 5e12
    # a short pressure time constant so that the scaling is far from 1
    baro = dict(barostat=G.PDGPU_BERENDSEN_BAROSTAT, target_pressure=1.0, pressure_tau=20e-15, compress=4.6e-5)
    pos = e.get_positions()
    vel = v0.copy()
    fold = np.zeros_like(pos)
    box = s.box.astype(np.float64).copy()
    for st in range(2):
        print(f"case barostat {integ} step {st}", flush=True)
        f, en = e.compute(comps)
        md = G.MDParams(integrator=I, components=comps, timestep=dt, temperature=300.0, fric_coeff=gamma,
                        update_nlist=10, step_offset=st, total_steps=3, seed=seed, **baro)
        ep, ek = e.md(md, 1)
        if integ == "vv":
            O.vv_kick(s.mass, dt, f, vel)
        elif integ == "beeman":
            O.beeman_kick(s.mass, dt, st, f, vel)
        else:  # the kick alone: a last step does not move
            O.langevin_step(s.mass, dt, gamma, 300.0, st, st + 1, f, np.zeros((s.n, 6)), pos, vel)
        K = O.kinetic_energy(s.mass, vel)
        P = O.pressure(K, en["virial"], box)
        fac = O.berendsen_barostat(P, dt, 4.6e-5, 1.0, 20e-15, pos, box)
        if integ == "vv":
            O.vv_move(s.mass, dt, f, pos, vel)
        elif integ == "beeman":
            O.beeman_move(s.mass, dt, st, 3, f, fold, pos, vel)
        else:  # the move alone: step 0 does not kick
            noise = np.array([O.langevin_noise(seed, 0, st, i) for i in range(s.n)])
            O.langevin_step(s.mass, dt, gamma, 300.0, 0, 3, f, noise, pos, vel)
        b, p = e.get_box()
        print(f"pressure {p:.3f} Bar (oracle {P:.3f}), factor {fac:.12f}", flush=True)
        assert abs(fac - 1.0) > 1e-9
        assert p == pytest.approx(P, rel=1e-11)
        np.testing.assert_allclose(b, box, rtol=1e-14)
        assert ek[0] == pytest.approx(K, rel=1e-13)
        np.testing.assert_allclose(e.get_positions(), pos, rtol=0, atol=1e-11)
        np.testing.assert_allclose(e.get_velocities(), vel, rtol=1e-9, atol=1e-9 * np.abs(vel).max())


def test_npt_run_contracts_a_dilute_box():
    """Beeman with the Berendsen thermostat and barostat on a box at 0.8 g/cm^3:
    the pressure is negative, so the box shrinks step by step; the run stays
    finite and the list follows the box through its rebuilds."""
    s = S.water_box(512, seed=9, density=0.8)
    e = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0, bonded=True)
    e.md(G.MDParams(integrator=G.PDGPU_LANGEVIN, components=G.PDGPU_NONBONDED | G.PDGPU_BONDED,
                    timestep=0.5e-15, temperature=300.0, fric_coeff=5e13, update_nlist=10, step_offset=0,
                    total_steps=1 << 30, seed=4), 200)
    e.set_initial_speeds(300.0, seed=2)
    b0 = e.get_box()[0].copy()
    md = G.MDParams(integrator=G.PDGPU_BEEMAN, components=G.PDGPU_NONBONDED | G.PDGPU_BONDED, timestep=1e-15,
                    temperature=300.0, update_nlist=10, step_offset=0, total_steps=301, seed=1,
                    thermostat=G.PDGPU_BERENDSEN, berendsen_tau=100e-15, barostat=G.PDGPU_BERENDSEN_BAROSTAT,
                    target_pressure=1.0, pressure_tau=2000e-15, compress=4.6e-5)
    ep, ek = e.md(md, 300)
    b1, p1 = e.get_box()
    print(f"box {b0[0]:.4f} -> {b1[0]:.4f} A, last pressure {p1:.1f} Bar", flush=True)
    assert np.isfinite(ep).all() and np.isfinite(ek).all()
    assert (b1 < b0).all() and np.allclose(b1 / b0, b1[0] / b0[0], rtol=1e-12)
    assert e.full_update_count() >= 30


def test_water_nve_runs_and_reports():
    s = S.water_box(1000, seed=12)
    e = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0, bonded=True)
    e.set_velocities(mb_velocities(s, 300.0, 5) * 0.1)
    md = G.MDParams(integrator=G.PDGPU_VELOCITY_VERLET, components=G.PDGPU_NONBONDED | G.PDGPU_BONDED,
                    timestep=0.5e-15, update_nlist=10, step_offset=0, total_steps=100, seed=1)
    ep, ek = e.md(md, 100)
    assert np.all(np.isfinite(ep)) and np.all(np.isfinite(ek))
    assert e.full_update_count() == 10


def test_fused_launches_equal_separate_ones():
    """The bonded terms run in the nonbonded kernel's last workgroups when both
    components are evaluated: the energies equal those of separate evaluations
    exactly and the forces to the rounding of adding two J/m arrays."""
    s = S.water_box(512, seed=9)
    e = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0, bonded=True)
    e.build_list()
    f, en = e.compute(G.PDGPU_NONBONDED | G.PDGPU_BONDED)
    fn, enn = e.compute(G.PDGPU_NONBONDED)
    fb, enb = e.compute(G.PDGPU_BONDED)
    for k in ("epot_vdw", "epot_elec"):
        assert en[k] == enn[k], k
    for k in ("epot_bond", "epot_angle", "epot_torsion"):
        assert en[k] == enb[k], k
    assert np.abs(f - (fn + fb)).max() <= 1e-14 * np.abs(f).max()


@pytest.mark.parametrize("integ", [G.PDGPU_BEEMAN, G.PDGPU_LANGEVIN, G.PDGPU_VELOCITY_VERLET])
def test_md_run_equals_single_step_calls(integ):
    """Inside one pdgpu_md call the integrator does the next step's opening work
    (slot positions, prune displacement, accumulator clears) and a step's energy
    sums run in the next step's nonbonded kernel; one-step calls do neither.  A
    25-step run (list rebuilt at steps 0, 10, 20) and 25 one-step calls give the
    same positions, velocities and energy trace, bit for bit."""
    s = S.water_box(512, seed=6)
    comps = G.PDGPU_NONBONDED | G.PDGPU_BONDED
    v0 = mb_velocities(s, 300.0, 3)
    runs = []
    for mode in ("run", "steps"):
        e = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0, bonded=True)
        e.set_velocities(v0)
        print(f"case integrator {integ} {mode}", flush=True)
        if mode == "run":
            md = G.MDParams(integrator=integ, components=comps, timestep=1e-15, temperature=300.0, fric_coeff=5e12,
                            update_nlist=10, step_offset=0, total_steps=25, seed=4)
            ep, ek = e.md(md, 25)
        else:
            ep, ek = np.zeros(25), np.zeros(25)
            for st in range(25):
                md = G.MDParams(integrator=integ, components=comps, timestep=1e-15, temperature=300.0,
                                fric_coeff=5e12, update_nlist=10, step_offset=st, total_steps=25, seed=4)
                a, b = e.md(md, 1)
                ep[st], ek[st] = a[0], b[0]
        runs.append((e.get_positions(), e.get_velocities(), ep, ek))
    (p1, v1, ep1, ek1), (p2, v2, ep2, ek2) = runs
    assert np.array_equal(p1, p2) and np.array_equal(v1, v2)
    assert np.array_equal(ep1, ep2) and np.array_equal(ek1, ek2)


@pytest.mark.parametrize("n_waters,thermo", [(1, G.PDGPU_BERENDSEN), (85, G.PDGPU_ANDERSEN), (86, G.PDGPU_BERENDSEN),
                                             (343, G.PDGPU_BERENDSEN), (1366, G.PDGPU_BERENDSEN)])
def test_thermostat_steps_share_launches(n_waters, thermo):
    """With a thermostat every workgroup of the moving kernel sums the kinetic-energy
    partials (one to 17 of them here) and opens the next step; one-step calls open
    theirs apart.  Same bits, and the first step's kinetic energy is the plain sum
    (FP64 sums of n positive terms in another order: n ulp at most)."""
    s = S.water_box(n_waters, seed=6)
    if n_waters < 343:
        s.box = None
    comps = G.PDGPU_NONBONDED | G.PDGPU_BONDED
    v0 = mb_velocities(s, 300.0, 3)
    runs = []
    for step_sizes in ([6], [1] * 6):
        e = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0, bonded=True)
        e.set_velocities(v0)
        print(f"case n={3 * n_waters} thermostat {thermo} calls {len(step_sizes)}", flush=True)
        ek = []
        for k in step_sizes:
            md = G.MDParams(integrator=G.PDGPU_BEEMAN, components=comps, timestep=1e-15, temperature=250.0,
                            thermostat=thermo, berendsen_tau=100e-15, andersen_rate=0.5, update_nlist=4,
                            step_offset=len(ek), total_steps=100, seed=4)
            ek += list(e.md(md, k)[1])
        runs.append((e.get_positions(), e.get_velocities(), np.array(ek)))
    for a, b in zip(*runs):
        assert np.array_equal(a, b)
    plain = 0.5 * (s.mass[:, None] * v0 ** 2).sum()
    assert abs(runs[0][2][0] - plain) <= 4 * s.n * np.finfo(float).eps * plain


def test_md_autotuner_restores_state():
    """pdgpu_autotune_md times MD steps at each prune margin from the same state,
    keeps the fastest and restores positions, velocities and the update count; the
    margin changes speed only (forces equal those at the default margin to FP32
    summation order); a second call with the same key reuses the choice."""
    s = S.water_box(512, seed=13)
    comps = G.PDGPU_NONBONDED | G.PDGPU_BONDED
    v0 = mb_velocities(s, 300.0, 2)
    md = G.MDParams(integrator=G.PDGPU_BEEMAN, components=comps, timestep=1e-15, update_nlist=10,
                    step_offset=0, total_steps=1000, seed=1)
    a = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0, bonded=True)
    a.set_velocities(v0)
    a.build_list()
    p0, v0d, n0 = a.get_positions(), a.get_velocities(), a.full_update_count()
    print("case autotune water 512", flush=True)
    m, ms = a.autotune_md(md, trial_steps=12, margins=[0.3, 0.6], retune=True)
    assert m in (0.3, 0.6) and ms is not None and np.all(ms > 0)
    assert np.array_equal(a.get_positions(), p0) and np.array_equal(a.get_velocities(), v0d)
    assert a.full_update_count() == n0
    m2, ms2 = a.autotune_md(md, trial_steps=12, margins=[0.3, 0.6])
    assert m2 == m and ms2 is None
    b = G.engine_for(s, G.nb_params(**WATER_NB), padding=2.0, bonded=True)
    b.set_velocities(v0)
    fa, ea = a.compute(comps)
    fb, eb = b.compute(comps)
    assert rel_rms(fa, fb) <= 1e-6
    assert ea["epot"] == pytest.approx(eb["epot"], rel=1e-6)
    ep, _ = a.md(md, 15)
    assert np.all(np.isfinite(ep))
