"""Benchmark: ns/day of NVE MD on the 98,304-atom TIP3P box (one MI355X).

Workload (the explicit-solvent configuration): 32,768 TIP3P waters on the even
lattice with uniformly random orientations (seeded), cubic box 99.346 A at
1.000 g/cm^3, orthogonal PBC, LJ + Coulomb cutoff 10 A with 8-10 A switching
(Coulomb force switch, LJ energy switch), list padding 2 A rebuilt every 10
steps, flexible TIP3P bonds/angle, PD's Beeman integrator (its default) at
1 fs.  A "step" is one MD step: the list refresh when due (cleanSpace +
rebuild), nonbonded + bonded forces and the FP64 integrator, all on the device.

Before timing, the lattice is relaxed by device Langevin dynamics (untimed) so
the NVE window starts from a physical state; the warmup steps are NVE, then the
autotuner picks the prune margin of the nonbonded list (each candidate timed over
--tune-steps steps from the same state, which is restored).  After
the timed window the same run continues --drift-steps NVE steps (untimed): the
energy drift is fitted over the timed and drift steps together.

Also measured: the list rebuild on its own (HBM roofline), and the GB/SA
workloads on AMBER99 chains (one 300-residue chain; 256 uneven chains batched
against the single-system engine looped over them; a 64-replica REMD batch).

Prints one JSON line (see the keys below).  `--gpus N` with N > 1 exits: this
build runs on one GPU.
"""
import argparse
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

FP32_PEAK_TFLOPS = 157.3     # MI355X FP32 vector/matrix peak (dense)
HBM_PEAK_GBPS = 8000.0       # MI355X HBM3E
# VALU issue ceiling: 256 CUs x 4 SIMDs, each 16 lanes wide, so a wave64 VALU
# instruction (FP32 without packing, or FP64) holds its SIMD for 4 cycles at the
# 2.4 GHz peak engine clock: 614 G wave instructions per second
VALU_SIMDS = 1024
ENGINE_HZ = 2.4e9
CYCLES_PER_VALU = 4
# Algorithmic FLOPs per unit of work, from PD's expression trees (add/sub/mul = 1,
# FMA = 2, sqrt/rcp/div = 1): a list entry tested and outside the cutoff, a pair
# at r <= InnerCutoff (LJ + force-switched Coulomb inner branch + accumulation),
# a pair in the switching shell (adds the LJ switch and the Coulomb polynomial).
FLOP_TESTED, FLOP_INNER, FLOP_SHELL = 11, 53, 81


def log(msg):
    print(msg, file=sys.stderr, flush=True)


def pair_classes(eng, box, cutoff, inner):
    """Counts of PD list entries by distance class at the current positions."""
    counts, packed = eng.get_pairs()
    pos = eng.get_positions()
    i = np.repeat(np.arange(len(counts)), counts)
    j = (packed & 0xFFFFFF).astype(np.int64)
    bo = (packed >> 24) & 7
    img = (packed >> 27).astype(np.int64)
    sh = np.stack([(img // 9) - 1, ((img // 3) % 3) - 1, (img % 3) - 1], axis=1) * box[None, :]
    n_tot = len(packed)
    in_cut = inner_cnt = 0
    step = 4_000_000
    for a in range(0, n_tot, step):
        b = min(n_tot, a + step)
        d = pos[j[a:b]] - pos[i[a:b]] + sh[a:b]
        r2 = (d * d).sum(axis=1)
        keep = (bo[a:b] >= 3)
        in_cut += int(((r2 <= cutoff * cutoff) & keep).sum())
        inner_cnt += int(((r2 <= inner * inner) & keep).sum())
    return n_tot, in_cut, inner_cnt


PMC_SUMMARY = os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles",
                           "water_box_98304_hbm_bytes.md")


FLOPS_SUMMARY = os.path.join(os.path.dirname(PMC_SUMMARY), "valu_flops_counters.md")


TIMING_EVERY = 7


def pmc_traffic(kernel):
    """HBM bytes per launch of `kernel` from the committed rocprofv3 --pmc summary
    (FETCH_SIZE and WRITE_SIZE runs of this bench, each scaled by what the counter
    reads for a copy of known size); {} when the summary is absent."""
    try:
        for line in open(PMC_SUMMARY):
            if line.startswith("PMC_JSON "):
                d = json.loads(line[len("PMC_JSON "):])
                if kernel in d:
                    return {"bytes_per_launch": d[kernel]["hbm_bytes_per_launch"],
                            "source": os.path.relpath(PMC_SUMMARY, os.path.dirname(PMC_SUMMARY) + "/..")}
    except OSError:
        pass
    return {}


def executed_flops(kernel, launch_s):
    """Issued FP32 VALU rate of `kernel` over a measured launch time: the FLOP per
    launch that the committed SQ-counter summary gives (64 lanes x (2 FMA + ADD +
    MUL + TRANS) instructions, lanes masked off included), against the FP32 peak;
    and the share of the VALU issue ceiling its instructions (all kinds) take
    over that time.  {} when the summary is absent."""
    try:
        for line in open(FLOPS_SUMMARY):
            if line.startswith("FLOPS_JSON "):
                d = json.loads(line[len("FLOPS_JSON "):])
                if kernel in d and launch_s > 0:
                    t = d[kernel]["fp32_flop_per_launch"] / launch_s / 1e12
                    issue = d[kernel]["valu_insts"] * CYCLES_PER_VALU / (VALU_SIMDS * ENGINE_HZ * launch_s)
                    return {"tflops": round(t, 3), "frac": round(t / FP32_PEAK_TFLOPS, 5),
                            "fp32_flop_per_launch": d[kernel]["fp32_flop_per_launch"],
                            "valu_insts_per_launch": d[kernel]["valu_insts"],
                            "valu_issue_frac": round(issue, 4),
                            "source": os.path.relpath(FLOPS_SUMMARY, os.path.dirname(FLOPS_SUMMARY) + "/..")}
    except OSError:
        pass
    return {}


def host_cpu():
    """(model name, logical CPUs of the host, CPUs this process may run on)."""
    model = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    try:
        avail = len(os.sched_getaffinity(0))
    except AttributeError:
        avail = os.cpu_count() or 1
    return model, os.cpu_count() or 1, avail


def baseline_threads():
    """Threads of the multi-core CPU baseline: every CPU this process may use, at
    most 16 (a one-GPU box's share of its host)."""
    return max(1, min(16, host_cpu()[2]))


def best_of(fn, reps=2):
    best, out = float("inf"), None
    for _ in range(reps):
        t0 = time.perf_counter()
        out = fn()
        best = min(best, time.perf_counter() - t0)
    return best, out


def cpu_baseline(sysw, nb_kw, padding, eng=None, comps=0):
    """The FP64 oracle (PD's algorithms restated in C) on the same box, on one
    thread and on every CPU of the process (OpenMP: per-thread force buffers summed
    in thread order): the list build with a cell grid (the pair set of PD's
    O(N^2) loop, which is timed once on one thread as well), the fast2 nonbonded
    forces, and the bonded forces + Beeman step (one thread in both).  `value`
    is the multi-core rate with the list amortised over the 10-step interval.

    With `eng`, the engine evaluates the same positions as well, and the result
    carries the error of the device forces and energy against the oracle: the
    error the headline number is stated at."""
    from oracle import oracle as O
    pos = O.clean_space(sysw)
    bo = O.bond_order(sysw)
    p = O.nb_params(**nb_kw)
    cut = max(p.Cutoff, p.VdwCutoff)
    basis = O.basis_vectors(True, sysw.box, cut)
    T = baseline_threads()
    model, ncpu, avail = host_cpu()
    t_n2, (counts, packed) = best_of(lambda: O.build_list(sysw, pos, cut, padding, False, bo), reps=1)
    rows = {}
    for th in (1, T):
        t_list, (c2, k2) = best_of(lambda: O.build_list(sysw, pos, cut, padding, False, bo, cells=True,
                                                        threads=th))
        assert np.array_equal(k2, packed), "cell-grid list differs from PD's all-pairs list"
        t_nb, (f, e_nb) = best_of(lambda: O.nb_forces(sysw, pos, counts, packed, p, basis, threads=th))

        def rest():
            fb, e_b = O.bonded_forces(sysw, pos)
            vel = np.zeros_like(pos)
            O.beeman_step(sysw.mass, 1e-15, 1, 3, f + fb, np.zeros_like(pos), pos.copy(), vel)
            return fb, e_b
        t_rest, (fb, e_b) = best_of(rest)
        per_step = t_list / 10.0 + t_nb + t_rest
        rows[th] = {"threads": th, "ns_per_day": round(86400.0 / per_step * 1e-6, 6),
                    "list_build_s": round(t_list, 4), "nonbonded_s": round(t_nb, 4),
                    "bonded_and_integrator_s": round(t_rest, 4), "s_per_step": per_step}
    out = {
        "value": rows[T]["ns_per_day"],
        "unit": "ns/day",
        "cores": T,
        "kind": "port",
        "cpu_model": model,
        "host_logical_cpus": ncpu,
        "cpus_available": avail,
        "sample": (f"oracle (PD's list build + fast2 nonbonded + bonded + Beeman, FP64) on the same {sysw.n}-atom "
                   f"box at the end of the timed run, {T} OpenMP threads on {model}: list (cell grid) "
                   f"{rows[T]['list_build_s']:.3f} s amortised over 10 steps, nonbonded {rows[T]['nonbonded_s']:.3f} s, "
                   f"bonded + integrator {rows[T]['bonded_and_integrator_s']:.3f} s (one thread)"),
        "by_threads": [{k: v for k, v in r.items() if k != "s_per_step"} for r in rows.values()],
        "pd_n2_list_build_s_1_thread": round(t_n2, 3),
        "value_1_thread_with_pd_list_build": round(86400.0 / (t_n2 / 10.0 + rows[1]["s_per_step"]
                                                              - rows[1]["list_build_s"] / 10.0) * 1e-6, 6),
    }
    if eng is not None:
        eng.set_positions(pos)
        eng.build_list()
        gf, ge = eng.compute(comps)
        fo = f + fb
        eo = e_nb["epot"] + e_b["epot"]
        terms = {k: e_nb[k] + e_b[k] for k in ("epot_vdw", "epot_elec", "epot_bond", "epot_angle")}
        out["error"] = {
            "force_rms_rel": float(np.sqrt(((gf - fo) ** 2).mean()) / np.sqrt((fo ** 2).mean())),
            "energy_rel": float(abs(ge["epot"] - eo) / abs(eo)),
            "per_term_rel": {k: float(abs(ge[k] - v) / abs(v)) for k, v in terms.items() if v != 0.0},
            "epot_kcal_mol": round(eo * 6.02214076e23 / 4184.0, 3),
            "reference": "FP64 oracle at the same positions (nonbonded + bonded)",
        }
    return out


def drift_fit(ep, ek, n_atoms, dt_fs=1.0):
    """Linear fit of the total energy over an NVE trace (J per step): the slope in
    kcal/mol/ns and per degree of freedom in kT/ns, the RMS about the fit, and the
    temperature at the start and the end."""
    from pd_amd import units as U
    etot = (np.asarray(ep) + np.asarray(ek)) * U.J_TO_KCALMOL
    t_ns = np.arange(len(etot)) * dt_fs * 1e-6
    slope, icpt = np.polyfit(t_ns, etot, 1)
    kt_kcal = U.KB * 300.0 * U.J_TO_KCALMOL
    temp = 2.0 * np.asarray(ek) / (3.0 * n_atoms * U.KB)
    return {"integrator": "beeman", "steps": int(len(etot)), "slope_kcal_mol_per_ns": float(slope),
            "slope_kT_per_dof_per_ns": float(slope / (3 * n_atoms * kt_kcal)),
            "etot_rms_about_fit_kcal_mol": float(np.std(etot - (slope * t_ns + icpt))),
            "etot_start_kcal_mol": float(etot[0]),
            "temperature_K": [round(float(temp[:10].mean()), 2), round(float(temp[-10:].mean()), 2)]}


def small_box_drift(G, S, nb_kw, padding, steps):
    """NVE drift of a 512-water box (1,536 atoms, the same force field and cutoffs)
    from one relaxed start: the device (FP32 pair math, fixed-point sums) and the
    FP64 oracle (PD's list, fast2 nonbonded, bonded and Beeman restated in C)
    each run `steps` Beeman steps at 1 fs.  The difference of the two slopes is
    what the device's arithmetic adds."""
    from oracle import oracle as O
    w = S.water_box(512, seed=6)
    comps = G.PDGPU_NONBONDED | G.PDGPU_BONDED
    e = G.engine_for(w, G.nb_params(**nb_kw), padding=padding, bonded=True)
    e.md(G.MDParams(integrator=G.PDGPU_LANGEVIN, components=comps, timestep=0.5e-15, temperature=300.0,
                    fric_coeff=5e13, update_nlist=10, step_offset=0, total_steps=1 << 30, seed=12), 300)
    e.set_initial_speeds(300.0, seed=6)
    pos = np.ascontiguousarray(e.get_positions())
    vel = np.ascontiguousarray(e.get_velocities())
    md = G.MDParams(integrator=G.PDGPU_BEEMAN, components=comps, timestep=1e-15, update_nlist=10,
                    step_offset=0, total_steps=steps + 1, seed=1)
    ep, ek = e.md(md, steps)
    dev = drift_fit(ep, ek, w.n)
    p = O.nb_params(**nb_kw)
    bo = O.bond_order(w)
    cut = max(p.Cutoff, p.VdwCutoff)
    basis = O.basis_vectors(True, w.box, cut)
    fold = np.zeros_like(pos)
    eo_p, eo_k = np.zeros(steps), np.zeros(steps)
    t0 = time.perf_counter()
    for st in range(steps):
        if st % 10 == 0:  # PD's refresh: cleanSpace, then a new list
            pos = np.ascontiguousarray(O.clean_space(w, pos))
            counts, packed = O.build_list(w, pos, cut, padding, False, bo, cells=True)
        f, en = O.nb_forces(w, pos, counts, packed, p, basis)
        fb, eb = O.bonded_forces(w, pos)
        eo_k[st] = O.beeman_step(w.mass, 1e-15, st, steps + 1, f + fb, fold, pos, vel)
        eo_p[st] = en["epot"] + eb["epot"]
    t_o = time.perf_counter() - t0
    orc = drift_fit(eo_p, eo_k, w.n)
    gap = np.abs((np.asarray(ep) + np.asarray(ek)) - (eo_p + eo_k)) * 6.02214076e23 / 4184.0
    return {"n_atoms": w.n, "steps": steps, "device": dev, "oracle_fp64": orc,
            "slope_difference_kcal_mol_per_ns": dev["slope_kcal_mol_per_ns"] - orc["slope_kcal_mol_per_ns"],
            "etot_gap_kcal_mol": {"step_100": float(gap[min(100, steps - 1)]), "max": float(gap.max())},
            "oracle_seconds": round(t_o, 2)}


GB_KW = dict(Cutoff=999.0, InnerCutoff=999.0, VdwCutoff=999.0, VdwInnerCutoff=999.0, GbsaStillCutoff=999.0,
             DielectricSolute=1.0, DielectricSolvent=78.5, Vdw14Scaling=0.5, Elec14Scaling=0.83333)
# algorithmic FLOPs per unordered pair and step of the three GB passes: pair pass 86,
# Born radii 2 x 16, chain rule 2 x 28 (174 in total)
GB_FLOP_PAIR, GB_FLOP_RADII, GB_FLOP_CHAIN = 86, 32, 56
GB_COMPS_NAMES = ("epot_pol", "epot_vdw", "epot_elec", "epot_surf", "epot_bond", "epot_angle", "epot_torsion")
SD_STEPS = 200  # steepest-descent relaxation of every built chain (on the device)


def _build_chain(args):
    from pd_amd import forcefield as F
    n_res, seed = args
    return F.random_peptide(n_res, seed)


def build_chains(specs, workers):
    if workers <= 1 or len(specs) < 4:
        return [_build_chain(s) for s in specs]
    import multiprocessing as mp
    with mp.get_context("fork").Pool(workers) as pool:
        return pool.map(_build_chain, specs, chunksize=max(1, len(specs) // (4 * workers)))


def gb_engine(G, s, seed, relax=True):
    """An AMBER99 GB/SA engine of chain `s` (LCPO with GlobalASP 0.005 updated
    every 5 steps), relaxed by SD_STEPS device steepest-descent steps, with
    Maxwell-Boltzmann velocities at 300 K."""
    from pd_amd import forcefield as F
    e = G.engine_for(s, None, bonded=True)
    e.setup_gb(G.gb_params(**GB_KW), s.gbrad, s.cov)
    use, rad, P = F.lcpo_params_ff(s)
    e.setup_lcpo(G.LCPOParams(GlobalASP=0.005, UpdateSasa=5), rad, P, use)
    if relax:
        e.minimise(G.min_params(G.PDGPU_GB | G.PDGPU_BONDED | G.PDGPU_SASA), SD_STEPS)
    e.set_initial_speeds(300.0, seed=seed)
    return e


def gb_oracle(s, pos, threads=0):
    """The FP64 oracle's GB/SA evaluation of chain `s` at `pos`: PD's list (all
    pairs, shadow, cell grid), Born radii, the FastMode pass (these three on
    `threads` OpenMP threads when > 0), bonded terms and LCPO (one thread).
    Returns (forces, energy terms, total, timings of list / GB / bonded / LCPO)."""
    from oracle import oracle as O
    from pd_amd import forcefield as F
    from pd_amd import units as U
    s2 = s.copy()
    s2.pos = pos
    p = O.gb_params(**GB_KW)
    bo = O.bond_order(s2)
    t0 = time.perf_counter()
    counts, packed = O.build_list(s2, pos, max(p.Cutoff, p.VdwCutoff), 0.5, True, bo, cells=True, threads=threads)
    t_list = time.perf_counter() - t0
    t0 = time.perf_counter()
    Vj, t123, _ = O.gb_fixed_terms(s2, p)
    born = O.gb_radii(s2, pos, Vj, t123, p, counts, packed, threads=threads)
    f_gb, e_gb = O.gb_forces_fast(s2, pos, Vj, born, p, counts, packed, threads=threads)
    t_gb = time.perf_counter() - t0
    t0 = time.perf_counter()
    f_b, e_b = O.bonded_forces(s2, pos)
    t_b = time.perf_counter() - t0
    use, rad, P = F.lcpo_params_ff(s2)
    sig = np.full(s2.n, 0.005 / U.NA / U.J2KCAL)
    t0 = time.perf_counter()
    f_l, _, e_l = O.lcpo_forces(pos, use, rad, P, sig, counts, packed)
    t_lcpo = time.perf_counter() - t0
    terms = {"epot_pol": e_gb["epot_pol"], "epot_vdw": e_gb["epot_vdw"], "epot_elec": e_gb["epot_elec"],
             "epot_surf": e_l, "epot_bond": e_b["epot_bond"], "epot_angle": e_b["epot_angle"],
             "epot_torsion": e_b["epot_torsion"]}
    return f_gb + f_b + f_l, terms, e_gb["epot"] + e_b["epot"] + e_l, (t_list, t_gb, t_b, t_lcpo)


def gb_error(gf, ge, fo, terms, eo):
    return {
        "force_rms_rel": float(np.sqrt(((gf - fo) ** 2).mean()) / np.sqrt((fo ** 2).mean())),
        "energy_rel": float(abs(ge["epot"] - eo) / abs(eo)),
        "per_term_rel": {k: float(abs(ge[k] - v) / abs(v)) for k, v in terms.items() if v != 0.0},
    }


def gb_cpu_baseline(G, s, e, comps):
    """The FP64 oracle on the chain's final positions, on one thread and on every
    CPU of the process, and the engine's forces and energy at the same positions
    against it.  A step: the list every 10 steps (PD's UpdateNList default), Born
    radii + FastMode pass + bonded every step, LCPO every 5 (UpdateSasa)."""
    pos = e.get_positions()
    T = baseline_threads()
    model, ncpu, avail = host_cpu()
    rows = {}
    for th in (1, T):
        best = None
        for _ in range(2):
            fo, terms, eo, tm = gb_oracle(s, pos, threads=th)
            best = tm if best is None else tuple(min(a, b) for a, b in zip(best, tm))
        t_list, t_gb, t_b, t_lcpo = best
        per_step = t_list / 10.0 + t_gb + t_b + t_lcpo / 5.0
        rows[th] = {"threads": th, "steps_per_s": round(1.0 / per_step, 3), "list_build_s": round(t_list, 4),
                    "gb_radii_and_pair_pass_s": round(t_gb, 4), "bonded_s": round(t_b, 4), "lcpo_s": round(t_lcpo, 4)}
    gf, ge = e.compute(comps)
    err = gb_error(gf, ge, fo, terms, eo)
    err["reference"] = "FP64 oracle at the same positions (GB FastMode + bonded + LCPO)"
    return {
        "value": rows[T]["steps_per_s"], "unit": "steps/s", "cores": T, "kind": "port", "cpu_model": model,
        "host_logical_cpus": ncpu, "cpus_available": avail,
        "sample": (f"oracle on the same {s.n}-atom chain, FP64, {T} OpenMP threads: list {rows[T]['list_build_s']:.3f} s "
                   f"(every 10 steps), Born radii + FastMode pass {rows[T]['gb_radii_and_pair_pass_s']:.3f} s, "
                   f"bonded {rows[T]['bonded_s']:.4f} s and LCPO {rows[T]['lcpo_s']:.3f} s (every 5 steps) "
                   f"on one thread"),
        "by_threads": list(rows.values()),
        "error": err,
    }


def remd_error(G, base, rb, comps, nsys):
    """Per-replica error of the device energies and forces against the FP64 oracle
    at each replica's final positions."""
    fb, eb = rb.compute(comps)
    rows = []
    for k in range(nsys):
        fo, terms, eo, _ = gb_oracle(base, rb.get_positions(k))
        rows.append(gb_error(fb[k], eb[k], fo, terms, eo))
    er = np.array([r["energy_rel"] for r in rows])
    fr = np.array([r["force_rms_rel"] for r in rows])
    worst = {k: max(r["per_term_rel"].get(k, 0.0) for r in rows) for k in GB_COMPS_NAMES}
    return {"energy_rel_max": float(er.max()), "energy_rel_median": float(np.median(er)),
            "force_rms_rel_max": float(fr.max()), "per_term_rel_max": worst,
            "energy_rel_per_replica": [float(f"{x:.3e}") for x in er],
            "reference": "FP64 oracle at each replica's final positions (GB FastMode + bonded + LCPO)"}


def gb_benchmarks(args, log):
    """The GB/SA workloads on AMBER99 chains built from random sequences (backbone
    phi/psi from N(-60, 10) / N(-45, 10) degrees) and relaxed by 200 device
    steepest-descent steps: one 300-residue chain, 256 uneven chains batched vs the
    single-system engine looped over them, and 64 REMD replicas."""
    import torch
    from pd_amd import engine as G
    comps = G.PDGPU_GB | G.PDGPU_BONDED | G.PDGPU_SASA
    lang = dict(integrator=G.PDGPU_LANGEVIN, components=comps, timestep=2e-15, temperature=300.0,
                fric_coeff=1e12, update_nlist=0, step_offset=0, total_steps=1 << 30, seed=3, noise_stream=0)
    workers = min(16, os.cpu_count() or 1)
    out = {}

    # --- single 300-residue chain (all pairs) ---------------------------------
    t0 = time.perf_counter()
    s = build_chains([(300, 7)], 1)[0]
    e = gb_engine(G, s, 1)
    split, tune_us = e.autotune_gb()  # the work split of the GB tile kernels, measured here
    log(f"autotuner (single chain): split {split.tolist()} (radii/pair/chain), us at 1/2/4: "
        f"{np.round(tune_us, 2).tolist()}")
    e.md(G.MDParams(**lang), 10)
    pairs = s.n * (s.n - 1) // 2
    e.set_timing(True)
    torch.cuda.synchronize()
    ts = time.perf_counter()
    e.md(G.MDParams(**dict(lang, step_offset=10)), args.gb_steps)
    torch.cuda.synchronize()
    wall = time.perf_counter() - ts
    kt = {k: e.kernel_time(k) for k in ("gb_radii", "gb_pair", "gb_chain", "lcpo")}
    e.set_timing(False)
    pair_us = kt["gb_pair"][0] / max(kt["gb_pair"][1], 1) * 1e3
    achieved = pairs * GB_FLOP_PAIR / (pair_us * 1e-6) / 1e12
    out["single_chain"] = {
        "workload": f"gbsa_amber99_random_chain_300res_{s.n}atoms", "n_atoms": s.n, "steps": args.gb_steps,
        "steps_per_s": round(args.gb_steps / wall, 2), "ms_per_step": round(wall * 1e3 / args.gb_steps, 4),
        "ns_per_day": round(args.gb_steps * 2e-6 * 86400 / wall, 3), "pairs": pairs,
        "kernel_us": {k: round(v[0] / max(v[1], 1) * 1e3, 2) for k, v in kt.items()},
        "autotune": {"split_radii_pair_chain": split.tolist(),
                     "launch_us_at_split_1_2_4": np.round(tune_us, 3).tolist()},
        "roofline_gb_pair": {"bound": "valu", "achieved": round(achieved, 3), "peak": FP32_PEAK_TFLOPS,
                             "unit": "TFLOP/s", "frac": round(achieved / FP32_PEAK_TFLOPS, 5),
                             "algorithmic_flop_per_launch": pairs * GB_FLOP_PAIR,
                             "executed": executed_flops("k_gb_pass pair (300-residue chain)", pair_us * 1e-6)},
    }
    log(f"single chain ({s.n} atoms): {out['single_chain']['steps_per_s']} steps/s "
        f"({time.perf_counter() - t0:.1f} s)")
    if not args.no_cpu_baseline:
        cb = gb_cpu_baseline(G, s, e, comps)
        out["single_chain"]["error"] = cb.pop("error")
        out["single_chain"]["cpu_baseline"] = cb
        log(f"single chain on the CPU oracle: {cb['value']} steps/s; force rms rel "
            f"{out['single_chain']['error']['force_rms_rel']:.2e}")
    del e

    # --- 256 uneven chains: batched vs looping the single-system engine --------
    rng = np.random.default_rng(2024)
    lengths = rng.integers(20, 121, args.gb_systems)
    t0 = time.perf_counter()
    chains = build_chains([(int(n), 1000 + k) for k, n in enumerate(lengths)], workers)
    log(f"built {len(chains)} chains ({sum(c.n for c in chains)} atoms) in {time.perf_counter() - t0:.1f} s")
    t0 = time.perf_counter()
    engines = [gb_engine(G, c, 100 + k) for k, c in enumerate(chains)]
    log(f"relaxed {len(engines)} chains ({SD_STEPS} SD steps each) in {time.perf_counter() - t0:.1f} s")
    batch = G.Batch(engines)
    bsplit, btune = batch.autotune_gb()
    log(f"autotuner (batch): split {bsplit.tolist()}, us at 1/2/4: {np.round(btune, 2).tolist()}")
    batch.md(G.MDParams(**lang), 5)
    torch.cuda.synchronize()
    ts = time.perf_counter()
    batch.md(G.MDParams(**dict(lang, step_offset=5)), args.gb_batch_steps)
    torch.cuda.synchronize()
    wall_b = time.perf_counter() - ts
    agg_b = len(chains) * args.gb_batch_steps / wall_b
    def loop(plain):
        # each system stepped in turn by its own single-system engine; plain: the
        # FP64 one-thread-per-atom GB comparator instead of the tiled kernels
        for en in engines:
            en.set_gb_plain(plain)
            en.md(G.MDParams(**lang), 2)  # warm
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for en in engines:
            en.md(G.MDParams(**dict(lang, step_offset=2)), args.gb_plain_steps)
        torch.cuda.synchronize()
        return len(chains) * args.gb_plain_steps / (time.perf_counter() - t0)
    agg_p = loop(True)
    agg_s = loop(False)
    pair_total = sum(c.n * (c.n - 1) // 2 for c in chains)
    out["batched_chains"] = {
        "workload": f"gbsa_amber99_{len(chains)}_chains_20-120res", "n_systems": len(chains),
        "n_atoms": int(sum(c.n for c in chains)), "pairs_per_step": int(pair_total),
        "batched_steps_per_s": round(agg_b, 1), "plain_loop_steps_per_s": round(agg_p, 1),
        "plain_loop": ("the plain single-system FP64 path: one thread per atom over every other atom, FP64 "
                       "arithmetic and per-atom FP64 sums (pdgpu_set_gb_plain), each system stepped in turn"),
        "speedup_vs_plain": round(agg_b / agg_p, 2),
        "single_engine_loop_steps_per_s": round(agg_s, 1),
        "speedup_vs_single_engine_loop": round(agg_b / agg_s, 2),
        "batched_ms_per_step": round(wall_b * 1e3 / args.gb_batch_steps, 3),
        "gflop_per_step": round(pair_total * (GB_FLOP_PAIR + GB_FLOP_RADII + GB_FLOP_CHAIN) / 1e9, 3),
        "autotune": {"split_radii_pair_chain": bsplit.tolist(),
                     "launch_us_at_split_1_2_4": np.round(btune, 3).tolist()},
    }
    log(f"batched: {agg_b:.1f} vs plain FP64 {agg_p:.1f} vs looped single engines {agg_s:.1f} aggregate steps/s")
    del batch, engines, chains

    # --- REMD: 64 replicas of a 60-residue chain, 300-500 K ------------------
    base = build_chains([(60, 77)], 1)[0]
    e0 = gb_engine(G, base, 0)
    base.pos = e0.get_positions()  # every replica starts from the relaxed chain
    del e0
    temps = 300.0 * (500.0 / 300.0) ** (np.arange(args.remd_replicas) / (args.remd_replicas - 1))
    reps = [gb_engine(G, base, 500 + k, relax=False) for k in range(args.remd_replicas)]
    rb = G.Batch(reps)
    rb.set_temperatures(temps)
    rsplit, rtune = rb.autotune_gb()
    torch.cuda.synchronize()
    ts = time.perf_counter()
    acc, att, fe = rb.remd(G.MDParams(**dict(lang, total_steps=args.remd_interval)), args.remd_rounds, 11)
    torch.cuda.synchronize()
    wall_r = time.perf_counter() - ts
    rates = [a / t if t else None for a, t in zip(acc[:-1].tolist(), att[:-1].tolist())]
    out["remd"] = {
        "workload": f"remd_amber99_{args.remd_replicas}x_{base.n}atoms_300-500K", "rounds": args.remd_rounds,
        "exchange_interval": args.remd_interval,
        "aggregate_steps_per_s": round(args.remd_replicas * args.remd_rounds * args.remd_interval / wall_r, 1),
        "acceptance": [round(r, 3) if r is not None else None for r in rates],
        "acceptance_mean": round(float(np.mean([r for r in rates if r is not None])), 4),
        "attempts_per_pair": [int(t) for t in att[:-1].tolist()],
        "autotune": {"split_radii_pair_chain": rsplit.tolist(),
                     "launch_us_at_split_1_2_4": np.round(rtune, 3).tolist()},
    }
    log(f"remd: {out['remd']['aggregate_steps_per_s']} aggregate steps/s, mean acceptance "
        f"{out['remd']['acceptance_mean']}")
    if not args.no_cpu_baseline:
        out["remd"]["error"] = remd_error(G, base, rb, comps, args.remd_replicas)
        log(f"remd error vs oracle: energy rel max {out['remd']['error']['energy_rel_max']:.2e}, "
            f"force rms rel max {out['remd']['error']['force_rms_rel_max']:.2e}")
    return out


def copy_probe(mib):
    """A plain copy of known size: the reference point that converts the HBM byte
    counters of a profiler run (FETCH_SIZE / WRITE_SIZE) into bytes."""
    import torch
    n = mib * (1 << 20) // 4
    src = torch.rand(n, device="cuda")
    dst = torch.empty_like(src)
    for _ in range(20):
        dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"copy_probe_bytes_read": n * 4, "copy_probe_bytes_written": n * 4, "launches": 20}),
          flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=1000)
    ap.add_argument("--warmup", type=int, default=50)
    ap.add_argument("--relax", type=int, default=300, help="untimed Langevin relaxation steps")
    ap.add_argument("--waters", type=int, default=32768)
    ap.add_argument("--drift-steps", type=int, default=1000, help="untimed NVE steps after the timed window")
    ap.add_argument("--list-builds", type=int, default=20, help="list rebuilds timed on their own")
    ap.add_argument("--tune-steps", type=int, default=60, help="MD steps per prune margin the autotuner times (0: off)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-gb", action="store_true", help="skip the GB/SA workloads")
    ap.add_argument("--gb-only", action="store_true", help="only the GB/SA workloads (for profiling)")
    ap.add_argument("--gb-steps", type=int, default=200)
    ap.add_argument("--gb-systems", type=int, default=256)
    ap.add_argument("--gb-batch-steps", type=int, default=100)
    ap.add_argument("--gb-plain-steps", type=int, default=20)
    ap.add_argument("--remd-replicas", type=int, default=64)
    ap.add_argument("--remd-rounds", type=int, default=20)
    ap.add_argument("--remd-interval", type=int, default=500)
    ap.add_argument("--copy-probe", type=int, default=0, metavar="MIB",
                    help="only run a plain device copy of MIB MiB 20 times (calibrates HBM byte counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU; --gpus {args.gpus} is not supported "
              f"(the multi-GPU decomposition is design-only)", file=sys.stderr)
        sys.exit(2)
    if args.copy_probe:
        copy_probe(args.copy_probe)
        return

    import torch
    from pd_amd import engine as G
    from pd_amd import systems as S
    from pd_amd import units as U

    assert torch.cuda.is_available(), "no GPU visible"
    if args.gb_only:
        print(json.dumps({"gbsa": gb_benchmarks(args, log)}), flush=True)
        return
    t0 = time.perf_counter()
    w = S.water_box(args.waters, seed=2024)
    nb_kw = dict(Cutoff=10.0, InnerCutoff=8.0, VdwCutoff=10.0, VdwInnerCutoff=8.0, ForceSwitch=1)
    padding = 2.0
    eng = G.engine_for(w, G.nb_params(**nb_kw), padding=padding, bonded=True)
    comps = G.PDGPU_NONBONDED | G.PDGPU_BONDED
    log(f"built {w.n} atoms, box {w.box[0]:.3f} A in {time.perf_counter() - t0:.1f} s")

    # untimed relaxation of the lattice (Langevin, 0.5 fs, strong friction)
    relax = G.MDParams(integrator=G.PDGPU_LANGEVIN, components=comps, timestep=0.5e-15, temperature=300.0,
                       fric_coeff=5e13, update_nlist=10, step_offset=0, total_steps=1 << 30, seed=11)
    if args.relax:
        eng.md(relax, args.relax)
    eng.set_initial_speeds(300.0, seed=5)  # setInitialSpeeds: Maxwell-Boltzmann at exactly 300 K
    log(f"relaxed {args.relax} steps")

    total = args.warmup + args.steps + args.drift_steps + 1  # no step of the run is Beeman's last
    nve = G.MDParams(integrator=G.PDGPU_BEEMAN, components=comps, timestep=1e-15, temperature=300.0,
                     fric_coeff=0.0, update_nlist=10, step_offset=0, total_steps=total, seed=1)
    ep_w, ek_w = eng.md(nve, args.warmup)
    # the prune margin: each candidate timed over a few steps from this state (restored
    # afterwards; the next step rebuilds the list anyway)
    nve.step_offset = args.warmup
    tune = {"prune_margin_A": 0.4, "tuned": False}
    if args.tune_steps > 0:
        margins = [0.3, 0.4, 0.5, 0.6]
        m, ms = eng.autotune_md(nve, trial_steps=args.tune_steps, margins=margins, retune=True)
        tune = {"prune_margin_A": m, "tuned": True, "trial_steps": args.tune_steps, "margins_A": margins,
                "ms_per_step": [round(float(v), 4) for v in ms]}
        log(f"autotuner (prune margin): {m} A; ms per step at {margins}: {tune['ms_per_step']}")
    # pair classes at the start of the timed window -> algorithmic FLOPs per nonbonded launch
    eng.build_list()
    n_tot, n_cut, n_inner = pair_classes(eng, w.box, nb_kw["Cutoff"], nb_kw["InnerCutoff"])
    flops = (n_tot - n_cut) * FLOP_TESTED + n_inner * FLOP_INNER + (n_cut - n_inner) * FLOP_SHELL
    log(f"list entries {n_tot}, in cutoff {n_cut}, inner {n_inner}; {flops / 1e9:.3f} GFLOP per nonbonded launch")

    nve.step_offset = args.warmup
    # HIP events around every launch of each timed kernel in a short window, or
    # every 7th in a long one: each event pair costs the queue a few microseconds,
    # and 7 is prime to the 10-step rebuild cycle, so the samples cover every phase
    every = 1 if args.steps < 20 * TIMING_EVERY else TIMING_EVERY
    eng.set_timing(True, every=every)
    torch.cuda.synchronize()
    ts = time.perf_counter()
    ep, ek = eng.md(nve, args.steps)
    torch.cuda.synchronize()
    te = time.perf_counter()
    nb_ms, nb_launch = eng.kernel_time("nonbonded")
    pr_ms, pr_launch = eng.kernel_time("prune")
    eng.set_timing(False)
    wall = te - ts
    ms_per_step = wall * 1e3 / args.steps
    ns_day = args.steps * 1.0 * 1e-6 * 86400.0 / wall
    nb_avg_s = nb_ms / max(nb_launch, 1) / 1e3
    achieved = flops / nb_avg_s / 1e12

    # the same NVE run continued, untimed, for the energy drift
    nve.step_offset = args.warmup + args.steps
    ep_d, ek_d = eng.md(nve, args.drift_steps)
    drift = drift_fit(np.concatenate([ep, ep_d]), np.concatenate([ek, ek_d]), w.n)
    log(f"NVE drift over {drift['steps']} Beeman steps: {drift['slope_kcal_mol_per_ns']:.1f} kcal/mol/ns "
        f"({drift['slope_kT_per_dof_per_ns']:.2e} kT/ns per degree of freedom), T {drift['temperature_K']}")

    # the list rebuild on its own: cleanSpace, cluster grid and sort, pair search
    eng.set_timing(True, every=1)
    for _ in range(args.list_builds):
        eng.build_list()
    lb_ms, lb_n = eng.kernel_time("list_build")
    ps_ms, ps_n = eng.kernel_time("pair_search")
    eng.set_timing(False)
    lb_s = lb_ms / max(lb_n, 1) / 1e3
    ps_s = ps_ms / max(ps_n, 1) / 1e3
    list_bytes = int(w.n * 24 + n_tot * 4)
    log(f"list rebuild {lb_s * 1e6:.1f} us (pair search {ps_s * 1e6:.1f} us): "
        f"{list_bytes / lb_s / 1e9:.0f} GB/s of algorithmic bytes")

    nb_traffic = pmc_traffic("k_nonbonded")
    out = {
        "metric": "ns/day @98k-atom water box; batched GB/SA steps/s vs plain, at stated error",
        "value": round(ns_day, 3),
        "unit": "ns/day",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32",
        "data": "synthetic",
        "config": {
            "workload": "tip3p_water_box_98304_nve",
            "n_atoms": w.n,
            "box_A": round(float(w.box[0]), 4),
            "cutoff_A": 10.0, "switch_A": [8.0, 10.0], "padding_A": padding, "update_nlist": 10,
            "timestep_fs": 1.0, "integrator": "beeman (PD's default), FP64",
            "pair_math": "FP32, FP64 displacement/cutoff test, int64 fixed-point forces",
            "parallelism": "single GPU",
        },
        "pair_interactions_per_s": round(n_cut * args.steps / wall, 1),
        "autotune": tune,
        "nve_drift_kcal_mol_per_ns": round(drift["slope_kcal_mol_per_ns"], 3),
        "nve_drift": {"water_98304": drift},
        "roofline": {
            "bound": "valu",
            "kernel": "k_nonbonded<force switch, vdw>",
            "achieved": round(achieved, 3),
            "peak": FP32_PEAK_TFLOPS,
            "unit": "TFLOP/s",
            "frac": round(achieved / FP32_PEAK_TFLOPS, 5),
            "traffic": nb_traffic.get("bytes_per_launch"),
            "traffic_source": nb_traffic.get("source"),
            "avg_launch_us": round(nb_avg_s * 1e6, 3),
            "launches_timed": nb_launch,
            "timed_every": every,
            "algorithmic_flop_per_launch": int(flops),
            "executed": executed_flops("k_nonbonded (water)", nb_avg_s),
            "list_entries": int(n_tot),
            "pairs_in_cutoff": int(n_cut),
        },
        "list_build": {
            "what": "one whole rebuild: cleanSpace, cluster grid and sort, pair search",
            "avg_us": round(lb_s * 1e6, 3),
            "rebuilds_timed": lb_n,
            "pair_search_avg_us": round(ps_s * 1e6, 3),
            "algorithmic_bytes": list_bytes,
            "algorithmic_bytes_rule": "24 B per atom read + 4 B per entry of PD's packed list",
            "achieved_GBps": round(list_bytes / lb_s / 1e9, 1),
            "peak_GBps": HBM_PEAK_GBPS,
            "hbm_frac": round(list_bytes / lb_s / 1e9 / HBM_PEAK_GBPS, 5),
            "pair_search_hbm_frac": round(list_bytes / ps_s / 1e9 / HBM_PEAK_GBPS, 5),
            "traffic": pmc_traffic("k_pair_search").get("bytes_per_launch"),
            "prune_avg_launch_us": round(pr_ms / max(pr_launch, 1) * 1e3, 3),
            "prune_launches_timed": pr_launch,
        },
    }
    if not args.no_cpu_baseline:
        log("timing the CPU baseline (oracle) and the error against it...")
        w_end = w.copy()
        w_end.pos = eng.get_positions()
        cb = cpu_baseline(w_end, nb_kw, padding, eng, comps)
        out["error"] = cb.pop("error")
        out["cpu_baseline"] = cb
        log(f"CPU baseline {cb['value']} ns/day; force rms rel {out['error']['force_rms_rel']:.2e}, "
            f"energy rel {out['error']['energy_rel']:.2e}")
        out["nve_drift"]["water_1536_vs_oracle"] = small_box_drift(G, S, nb_kw, padding, args.drift_steps)
    del eng
    if not args.no_gb:
        out["gbsa"] = gb_benchmarks(args, log)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
