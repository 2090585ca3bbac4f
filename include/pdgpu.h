/*
 * pdgpu.h -- C ABI of the MI355X (gfx950) nonbonded / GB-SA force engine for PD.
 *
 * One engine handle holds one molecular system resident in HBM together with
 * its neighbour list, and plays the parts of three PD objects:
 *   - the neighbour list, a WorkSpace component (neighbourlist.h:54-126,
 *     NeighbourList::calcNewList neighbourlist.cpp:222-244, with
 *     WorkSpace::cleanSpace workspace.cpp:371-380 run before each rebuild as
 *     ProtocolBase::refreshNeighborList does, protocolbase.cpp:135-144);
 *   - the forcefield components FF_NonBonded (nonbonded.h:62-231),
 *     FF_GeneralizedBorn_Still (gbff.h:123-203) and FF_Bonded (ffbonded.h), behind
 *     ForcefieldBase::calcForces / calcEnergies (forcefield.h:110-239);
 *   - the MolecularDynamics integrators (md.cpp:805-855 velocity Verlet,
 *     md.cpp:858-919 Beeman, md.cpp:923-1059 Langevin), its Berendsen and
 *     Andersen thermostats (md.cpp:579-660) and momentum removal
 *     (md.cpp:263-272) run as a device-resident loop.
 *
 * Conventions (all entry points):
 *   - PD units at the boundary: positions in Angstrom, forces in J/m, energies in
 *     J per molecule, masses in kg, velocities in m/s, per-atom LJ epsilon as
 *     sqrt(epsilon[J]) (ffparam.cpp:1216), radius = R_min/2 in Angstrom.
 *   - Coordinate arrays are AoS xyz doubles with a caller-given byte stride, so
 *     PD's SnapShotAtom array (p, f, v dvectors, stride 72 bytes, snapshot.h:33-39)
 *     can be passed without copying into a temporary.
 *   - Every call returns PDGPU_OK (0) or a negative error code; the text of the
 *     last error of a handle is pdgpu_last_error(handle).  No C++ exception
 *     crosses this interface.  One handle is used by one host thread at a time.
 */
#ifndef PDGPU_H
#define PDGPU_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define PDGPU_OK 0
#define PDGPU_ERR_ARG (-1)      /* invalid argument or call order */
#define PDGPU_ERR_HIP (-2)      /* HIP runtime error */
#define PDGPU_ERR_SETUP (-3)    /* configuration PD itself rejects (e.g. >32 image vectors) */
#define PDGPU_ERR_NOMEM (-4)    /* device allocation failed */
#define PDGPU_ERR_UNSTABLE (-5) /* NaN energy: ProtocolBase::assertStability (protocolbase.cpp:126-132) */
#define PDGPU_ERR_CAPACITY (-6) /* the neighbour list does not fit: more candidates than 64 search passes hold */

typedef struct pdgpu_engine pdgpu_engine;

/* Energies of one evaluation; members mirror PD's Hamiltonian (hamiltonian.h:40-66). */
typedef struct pdgpu_energies {
  double epot;
  double epot_vdw;
  double epot_elec;
  double epot_pol;
  double epot_pol_self;
  double epot_pol_cross;
  double epot_bond;
  double epot_angle;
  double epot_torsion;
  double epot_surf;
  double virial; /* InternalVirial, sum of r * dE/dr [J] */
  double ekin;
} pdgpu_energies;

/* FF_NonBonded public parameters (nonbonded.h:72-143; defaults nonbonded.cpp:985-1021). */
typedef struct pdgpu_nb_params {
  double Cutoff, InnerCutoff, VdwCutoff, VdwInnerCutoff;
  double Vdw14Scaling, Elec14Scaling;
  double Dielectric, DDDielectricAlpha;
  int32_t DoVdw, DoElec, ForceSwitch, EnergySwitch;
  int32_t VdwCor;
  double VdwCorDensity, VdwCorEpsilon, VdwCorRadius, VdwCorCutoff;
} pdgpu_nb_params;

/* FF_GeneralizedBorn_Still parameters (gbff.cpp:34-55) and its inherited
 * nonbonded cutoffs and 1-4 scalings. */
typedef struct pdgpu_gb_params {
  double Cutoff, InnerCutoff, VdwCutoff, VdwInnerCutoff;
  double Vdw14Scaling, Elec14Scaling;
  double DielectricSolute, DielectricSolvent;
  double GbsaStillCutoff, ExpApproxThreshold, DielectricOffset, BornRadiusOffset;
  double P1, P2, P3, P4, P5;
  /* FF_GeneralizedBorn_Still::FastMode (PD default 1: calcForcesIncludingVacuo);
   * 0: FF_NonBonded::calcForces + calcBornForces (gbff.cpp:186-196, 1189-1437),
   * whose polarisation energy goes into epot only, as PD adds it. */
  int32_t FastMode;
} pdgpu_gb_params;

/* Component selection for pdgpu_compute / pdgpu_md. */
#define PDGPU_NONBONDED 0x1u /* FF_NonBonded::calcForces */
#define PDGPU_BONDED 0x2u    /* FF_Bonded bonds + angles + torsions */
#define PDGPU_GB 0x4u        /* FF_GeneralizedBorn_Still::calcForces (FastMode) */
#define PDGPU_SASA 0x8u      /* FF_SASA_LCPO::calcForces */
/* With PDGPU_ENERGY_ONLY the selected components run calcEnergies() instead of
 * calcForces() (ForcefieldBase::calcEnergies, forcefield.h:110-239): no forces
 * (f_accum must be NULL); FF_NonBonded::calcEnergies_Full (nonbonded.cpp:1184-1202),
 * FF_GeneralizedBorn_Still::calcEnergies (gbff.cpp:178-183, exact GB, no
 * FastMode swap), FF_SASA_LCPO::calcLCPOSasaEnergies (lcpo.cpp:453-560); FF_Bonded
 * energies are those of its force routine. */
#define PDGPU_ENERGY_ONLY 0x100u

/* Integrators of MolecularDynamics (md.h:76). */
#define PDGPU_VELOCITY_VERLET 1
#define PDGPU_BEEMAN 2 /* PD's default integrator (md.cpp:60) */
#define PDGPU_LANGEVIN 3

/* Thermostats of MolecularDynamics (md.h:96); they act in velocity Verlet and
 * Beeman steps (Langevin regulates the temperature itself). */
#define PDGPU_NO_THERMOSTAT 0
#define PDGPU_ANDERSEN 1
#define PDGPU_BERENDSEN 2

/* MolecularDynamics::Barostat (md.cpp:663-684) */
#define PDGPU_NO_BAROSTAT 0
#define PDGPU_BERENDSEN_BAROSTAT 1

typedef struct pdgpu_md_params {
  int32_t integrator;     /* PDGPU_VELOCITY_VERLET, PDGPU_BEEMAN or PDGPU_LANGEVIN */
  uint32_t components;    /* PDGPU_* forcefield components evaluated each step */
  double timestep;        /* s (MolecularDynamics::Timestep) */
  double temperature;     /* K (target temperature: Langevin and the thermostats) */
  double fric_coeff;      /* 1/s (MolecularDynamics::FricCoeff) */
  int32_t update_nlist;   /* MolecularDynamics::UpdateNList (list rebuild period) */
  int32_t step_offset;    /* first step number (Langevin's first/last step guards) */
  int32_t total_steps;    /* MolecularDynamics::Steps */
  uint64_t seed;          /* Langevin / Andersen noise: Philox4x32-10 key */
  uint32_t noise_stream;  /* Philox counter word 2; a batch adds the system index */
  int32_t thermostat;     /* MolecularDynamics::Thermostat: PDGPU_NO_THERMOSTAT (default), ... */
  int32_t remove_momentum; /* UpdateRemoveTotalMomentum (PD: 200); only with a thermostat, md.cpp:263-272 */
  double berendsen_tau;   /* s (BerendsenTau, PD: 100e-15) */
  double andersen_rate;   /* AndersenRate (PD: 0.1) */
  /* Berendsen barostat (md.cpp:537-552, 677-684), PeriodicBox only: after the
   * kick, P = (2 ekin - InternalVirial) / (3 V) in Bar, and every position and
   * the box are scaled by (1 + dt Compress (P - TargetPressure) / tau)^(1/3). */
  int32_t barostat;         /* PDGPU_NO_BAROSTAT (default) or PDGPU_BERENDSEN_BAROSTAT */
  double target_pressure;   /* Bar (TargetPressure, PD: 1) */
  double pressure_tau;      /* s (BerendsenPressureTau, PD: 2000e-15) */
  double compress;          /* 1/Bar (Compress, PD: 4.6e-5) */
  /* ProtocolBase::UpdateTra: after each step with every(step, UpdateTra)
   * (md.cpp:277, protocolbase.cpp:251-257) the positions and energy terms are
   * kept on the device as a frame for the caller's trajectory writers
   * (WorkSpace::outtra); pdgpu_get_frames returns them.  0: none. */
  int32_t update_tra;
} pdgpu_md_params;

/* ---- lifecycle -------------------------------------------------------------- */

/* Creates an engine for n_atoms atoms on HIP device `device`. */
int pdgpu_create(int32_t n_atoms, int32_t device, pdgpu_engine **out);
int pdgpu_destroy(pdgpu_engine *e);
const char *pdgpu_last_error(const pdgpu_engine *e);
/* Library build string (gfx target, compile flags); never NULL. */
const char *pdgpu_version(void);

/* ---- system description (ForcefieldBase::setup time) ------------------------- */

/* Per-atom Particle parameters (fundamentals.h:192-195) and masses. */
int pdgpu_set_atom_params(pdgpu_engine *e, const double *radius, const double *epsilon,
                          const double *charge, const double *mass);

/* Molecules as inclusive atom ranges (MoleculeBase::mol[i].ifirst/ilast), used
 * by WorkSpace::cleanSpace before each list rebuild. */
int pdgpu_set_molecules(pdgpu_engine *e, int32_t n_mol, const int32_t *first,
                        const int32_t *last);

/* BondOrder data (bondorder.h:60-124): the band matrix getDiagData() of
 * max_index_delta*(n-1) chars, and the off-diagonal partners of getOffDiagData()
 * flattened as (i, j, order) triples in PD's order. */
int pdgpu_set_bond_order(pdgpu_engine *e, int32_t max_index_delta, const int8_t *band,
                         int32_t n_sparse, const int32_t *sp_i, const int32_t *sp_j,
                         const int32_t *sp_order);

/* Convenience: BondOrder::reinit (bondorder.cpp:94-212) from covalent 1-2/1-3/1-4
 * partner lists in CSR form and residue indices, then pdgpu_set_bond_order. */
int pdgpu_set_bond_order_from_cov(pdgpu_engine *e, const int32_t *resid,
                                  const int32_t *off12, const int32_t *idx12,
                                  const int32_t *off13, const int32_t *idx13,
                                  const int32_t *off14, const int32_t *idx14);

/* Space: periodic != 0 gives an orthogonal PeriodicBox of edge lengths box[3]
 * centred on the origin (space.h:183-327); periodic == 0 gives InfiniteSpace. */
int pdgpu_set_space(pdgpu_engine *e, int32_t periodic, const double *box);
/* The current box edge lengths (PeriodicBox::boxSize, changed by a barostat) and
 * the pressure (Bar) of the last barostat step (MolecularDynamics::m_CurPress). */
int pdgpu_get_box(pdgpu_engine *e, double *box, double *pressure);

/* NeighbourListBase::requestCutoff / setPadding / calcShadow (neighbourlist.h:64-70). */
int pdgpu_request_cutoff(pdgpu_engine *e, double cutoff);
int pdgpu_set_padding(pdgpu_engine *e, double padding);
int pdgpu_calc_shadow(pdgpu_engine *e, int32_t enabled);

/* FF_NonBonded::setup (nonbonded.cpp:1025-1053): stores the parameters and
 * requests max(Cutoff, VdwCutoff) from the list.  Fails with PDGPU_ERR_SETUP
 * where FF_NonBonded::setupBasisVectors throws (more than 32 image vectors). */
int pdgpu_setup_nonbonded(pdgpu_engine *e, const pdgpu_nb_params *p);

/* FF_Bonded terms; force constants in PD units (J/A^2, J/rad^2, J), angles in rad.
 * Torsions carry up to 4 Fourier terms each (vn/nn/gamma are 4 per torsion). */
int pdgpu_set_bonded(pdgpu_engine *e, int32_t nb, const int32_t *bi, const int32_t *bj,
                     const double *bl, const double *bk, int32_t na, const int32_t *ai,
                     const int32_t *aa, const int32_t *aj, const double *theta0,
                     const double *ak, int32_t nt, const int32_t *ti, const int32_t *ta,
                     const int32_t *tb, const int32_t *tj, const int32_t *terms,
                     const double *vn, const double *nn, const double *gamma);

/* FF_GeneralizedBorn_Still::setup (gbff.cpp:57-104): GB radius of each atom's
 * type and the 1-2 / 1-3 partner lists with their equilibrium distances
 * (Particle::cov12atom/cov13atom, fundamentals.h:80-90).  The fixed Born terms
 * (calcFixedBornRadiiTerms, gbff.cpp:324-398) are computed here in FP64. */
int pdgpu_setup_gb(pdgpu_engine *e, const pdgpu_gb_params *p, const double *gbradius,
                   const int32_t *off12, const int32_t *idx12, const double *d12,
                   const int32_t *off13, const int32_t *idx13, const double *d13);

/* Work split of the GB passes (Born radii, pair terms, chain rule): split[k]
 * wavefronts share a task of pass k (one or two 64-atom i tiles against a run of j
 * tiles), taking its chunks of 16 rotated j steps in turn (1, 2 or 4; NULL: all 1;
 * until it is called, the number that suits the number of tasks).  Sums beyond a
 * chunk are integers, so forces and radii are the same bits for every split; energies
 * differ by FP64 rounding.  No counterpart in PD: the launch shape of the GB passes. */
int pdgpu_set_gb_split(pdgpu_engine *e, const int32_t *split);
/* The autotuner: one full GB pass on the current positions, then each tile kernel
 * 5 times at split 1, 2 and 4 (HIP events); keeps the fastest split per kernel,
 * returned in split[3]; us[9] (may be NULL) gets the average launch times,
 * us[3*k + m] for kernel k at split 1 << m.  Evaluate again afterwards: the force
 * accumulators hold the tuning launches.  The choice is kept for the process per
 * (atoms, systems, FastMode): a GB component set up later with that shape (an
 * engine or a batch) starts with it. */
int pdgpu_autotune_gb(pdgpu_engine *e, int32_t *split, double *us);
/* The plain comparator for the FastMode passes (on != 0): one thread per atom over
 * every other atom, FP64 arithmetic and FP64 per-atom sums, no tiles -- the
 * straightforward single-system GPU path the tiled and batched kernels are
 * measured against.  Same results within FP64 rounding; forces only. */
int pdgpu_set_gb_plain(pdgpu_engine *e, int32_t on);

/* FF_SASA_LCPO public parameters (lcpo.h:59-68). */
typedef struct pdgpu_lcpo_params {
  double GlobalASP;   /* atomic solvation parameter, kcal/mol/A^2 (lcpo.cpp:63) */
  int32_t UpdateSasa; /* full recalculation every UpdateSasa MD steps (lcpo.cpp:196-201) */
} pdgpu_lcpo_params;

/* FF_SASA_LCPO::setup (lcpo.cpp:33-127) with the per-atom result of its
 * LCPOSASATYPE lookup (readLCPOSection, lcpo.cpp:321-437): radius (the table
 * radius; 1.4 A is added here), P1..P4 (4 per atom), use (0 for hydrogens).
 * asp: per-atom solvation parameter in kcal/mol/A^2, or NULL for GlobalASP on
 * every atom. */
int pdgpu_setup_lcpo(pdgpu_engine *e, const pdgpu_lcpo_params *p, const double *radius, const double *P,
                     const int8_t *use, const double *asp);

/* Per-atom SASA (A^2) of the last full LCPO calculation (SASA_Atom::SASA). */
int pdgpu_get_sasa(pdgpu_engine *e, double *sasa);

/* ---- state ------------------------------------------------------------------ */

int pdgpu_set_positions(pdgpu_engine *e, const double *xyz, size_t stride_bytes);
int pdgpu_get_positions(pdgpu_engine *e, double *xyz, size_t stride_bytes);
int pdgpu_set_velocities(pdgpu_engine *e, const double *xyz, size_t stride_bytes);
int pdgpu_get_velocities(pdgpu_engine *e, double *xyz, size_t stride_bytes);

/* ---- neighbour list ----------------------------------------------------------- */

/* WorkSpace::cleanSpace then NeighbourList::calcNewList on the device
 * (protocolbase.cpp:135-144).  Positions held by the engine are moved the way
 * cleanSpace moves PD's. */
int pdgpu_build_list(pdgpu_engine *e);

/* NeighbourListBase::getFullUpdateCount (neighbourlist.h:71). */
int pdgpu_full_update_count(pdgpu_engine *e, uint32_t *count);

/* The pair set of the last build in PD's packed form (neighbourlist.h:131-151):
 * per-atom counts and entries j | bondorder<<24 | image<<27, atom after atom,
 * ascending j within an atom.  pdgpu_get_pair_count gives the total first. */
int pdgpu_get_pair_count(pdgpu_engine *e, int64_t *total);
int pdgpu_get_pairs(pdgpu_engine *e, int32_t *counts, uint32_t *packed, int64_t capacity);

/* ---- force evaluation ---------------------------------------------------------- */

/* Evaluates the selected components on the current positions, ADDS the forces
 * (J/m) into f_accum (stride as above; may be NULL) and writes the components'
 * energies (J) to *energies (may be NULL). */
int pdgpu_compute(pdgpu_engine *e, uint32_t components, double *f_accum, size_t stride_bytes,
                  pdgpu_energies *energies);

/* Allocation-free variant of pdgpu_compute.  It has no counterpart in PD; it is
 * for callers that cannot allocate device memory (code under stream capture,
 * tight serving loops, harnesses that forbid hipMalloc).  It calls no hipMalloc,
 * hipFree or allocating library routine:
 *   - components: PDGPU_NONBONDED and/or PDGPU_BONDED, optionally with
 *     PDGPU_ENERGY_ONLY (then d_f_accum must be NULL);
 *   - with PDGPU_NONBONDED the neighbour list must have been built
 *     (pdgpu_build_list sizes every buffer an evaluation writes); it is not
 *     rebuilt here;
 *   - forces are ADDED, in J/m, to d_f_accum, a DEVICE array of the caller with
 *     a byte stride (a multiple of 8, at least 24; PD's 72-byte SnapShotAtom
 *     stride works); may be NULL;
 *   - energies (J) as pdgpu_compute; may be NULL.
 * The energy partials live in one 1 MiB device array per GPU (131,072
 * doubles): systems whose partials need more (about 1 M atoms of nonbonded
 * work groups) are rejected with PDGPU_ERR_ARG.  All engines on one GPU share
 * that array, so calls on one GPU that overlap in time race. */
int pdgpu_compute_noalloc(pdgpu_engine *e, uint32_t components, double *d_f_accum, size_t stride_bytes,
                          pdgpu_energies *energies);

/* Born radii of the last GB evaluation (calcBornRadii_PairwiseApprox), Angstrom. */
int pdgpu_get_born_radii(pdgpu_engine *e, double *radii);

/* FF_NonBonded::calcEnergies with UsePartialRecalc (nonbonded.cpp:1154-1181,
 * 76-386), the energy path of Monte Carlo moves: the nonbonded energy at the
 * current positions from the energy of the previous call, re-evaluating only the
 * pairs that touch atoms whose position changed since then.  The first call, a
 * call after a list rebuild (a new full-update count) or a new system
 * description, and a call with more than 256 moved atoms evaluate the whole
 * energy.  components must be PDGPU_NONBONDED; fills epot, epot_vdw, epot_elec. */
int pdgpu_energy_update(pdgpu_engine *e, uint32_t components, pdgpu_energies *energies);

/* ---- molecular dynamics ----------------------------------------------------------- */

/* Runs n_steps steps of MolecularDynamics::run_core (md.cpp:219-284) on the
 * device: list refresh every update_nlist steps, force evaluation, integrator.
 * If epot_trace / ekin_trace are non-NULL they receive one value per step (J):
 * the potential energy of the step's force evaluation and the kinetic energy the
 * integrator computes.  Returns PDGPU_ERR_UNSTABLE if an energy became NaN.
 * Beeman's old forces (PD's oldatom[i].f) live in the engine across calls and
 * start at zero. */
int pdgpu_md(pdgpu_engine *e, const pdgpu_md_params *p, int32_t n_steps, double *epot_trace,
             double *ekin_trace);

/* The frames of the last pdgpu_md call (update_tra): up to max_frames frames of
 * positions (xyz: max_frames * n_atoms * 3 doubles, AoS, A), their step numbers
 * and energy terms (either may be NULL); *n_frames gets the number recorded. */
int pdgpu_get_frames(pdgpu_engine *e, int32_t max_frames, double *xyz, int32_t *steps,
                     pdgpu_energies *energies, int32_t *n_frames);

/* SnapShot::writeMIME / readMIME (snapshot.cpp:345-466): the checkpoint format of
 * PD's WorkSpace: "!PSP name", then 128 header bytes (atoms, epot in J, four
 * status words) and per atom p, v, f (FP64; A, m/s, J/m) in PD's 6-bit text
 * encoding (tools/io.cpp:95-178), then "!ENDPSP".  Writing takes the positions,
 * velocities and the forces and epot of the last evaluation; append != 0 adds to
 * the file.  Reading the named entry ("" = the first) sets positions and velocities. */
int pdgpu_write_snapshot(pdgpu_engine *e, const char *path, const char *name, int32_t append);
int pdgpu_read_snapshot(pdgpu_engine *e, const char *path, const char *name);

/* No counterpart in PD (an autotuner of this engine): the nonbonded kernel reads
 * a pruned copy of the list holding the pairs within Cutoff + margin at the last
 * prune, pruned again on the device once twice the largest displacement since
 * then reaches the margin (default 0.4 A).  Every margin gives PD's pair set; the
 * margin trades prunes against force-kernel work.  pdgpu_autotune_md runs
 * trial_steps steps of the protocol p (its components must include
 * PDGPU_NONBONDED and not PDGPU_SASA) at each of n_margins margins (NULL or 0:
 * 0.3, 0.4, 0.5, 0.6 A), each from the same state, keeps the fastest (the margin
 * in use stays unless another is more than 1% faster) and restores
 * positions, velocities, Beeman's old forces and the box; the next evaluation
 * rebuilds the list, so call it where the protocol's next step rebuilds anyway
 * (step % UpdateNList == 0).  *chosen (may be NULL) receives the margin kept, ms
 * (may be NULL, n_margins values) the milliseconds per step at each.  The choice
 * is kept for the process per (atoms, list cutoff, padding, space): later calls
 * with that key apply it without trials unless retune != 0.
 * pdgpu_set_prune_margin sets the margin directly. */
int pdgpu_autotune_md(pdgpu_engine *e, const pdgpu_md_params *p, int32_t trial_steps, int32_t n_margins,
                      const double *margins, int32_t retune, double *chosen, double *ms);
int pdgpu_set_prune_margin(pdgpu_engine *e, double margin);

/* MolecularDynamics::setInitialSpeeds (md.cpp:359-380): every atom's velocity
 * drawn from N(0, kB T / m) per component (PD's two Box-Muller calls, the second
 * overwriting vy, with Philox4x32-10 uniforms keyed by `seed` instead of glibc
 * rand()), then all scaled so that the kinetic energy is exactly 3 N kB T / 2
 * (setKineticEnergyTo, md.cpp:563-577). */
int pdgpu_set_initial_speeds(pdgpu_engine *e, double temperature, uint64_t seed, uint32_t noise_stream);

/* ---- minimisation ------------------------------------------------------------------ */

/* Minimisation parameters (minimise.h; defaults minimise.cpp:51-58). */
typedef struct pdgpu_min_params {
  uint32_t components;  /* PDGPU_* forcefield components evaluated each step */
  double step_size;     /* Minimisation::StepSize (PD: 2e5), A per J/m at multiplier 1 */
  int32_t update_nlist; /* list rebuild period (nonbonded component) */
} pdgpu_min_params;

/* Minimisation::runcore with Algorithm = SteepestDescent (minimise.cpp:111-252)
 * on the device: each step evaluates the forces and takes PD's descent step
 * (accept: multiplier x 1.2 and move along the force; reject: multiplier
 * x 0.5/1.2, positions restored, reference energy + 1 J).  The final positions
 * are the last accepted ones.  epot_trace (may be NULL) receives each step's
 * energy (J). */
int pdgpu_minimise(pdgpu_engine *e, const pdgpu_min_params *p, int32_t n_steps, double *epot_trace);

/* ---- batches of independent systems / REMD replicas ------------------------------ */

/* Many independent systems of uneven size advanced together on one GPU.  PD has
 * no batch object: its REX_Local (remd.h:127) runs replicas one after another on
 * one WorkSpace and its protocols run one system at a time; a batch holds N such
 * systems at once.  It is built from single-system engines that carry the full
 * setup (atom parameters, bond orders, bonded terms, GB, positions, velocities);
 * their data are copied, the engines stay usable.  GB parameters must be equal.
 * Systems keep their order; per-system arrays below are indexed by it. */
typedef struct pdgpu_batch pdgpu_batch;

int pdgpu_batch_create(int32_t n_systems, pdgpu_engine *const *systems, pdgpu_batch **out);
int pdgpu_batch_destroy(pdgpu_batch *b);
const char *pdgpu_batch_last_error(const pdgpu_batch *b);
/* Target temperature of each system (K); default 300. */
int pdgpu_batch_set_temperatures(pdgpu_batch *b, const double *temperatures);
/* pdgpu_set_gb_split / pdgpu_autotune_gb for a batch (all its systems' tile pairs
 * in one launch); the recorded step graph is redone with the new split. */
int pdgpu_batch_set_gb_split(pdgpu_batch *b, const int32_t *split);
int pdgpu_batch_autotune_gb(pdgpu_batch *b, int32_t *split, double *us);
int pdgpu_batch_get_positions(pdgpu_batch *b, int32_t system, double *xyz, size_t stride_bytes);
int pdgpu_batch_set_positions(pdgpu_batch *b, int32_t system, const double *xyz, size_t stride_bytes);
int pdgpu_batch_get_velocities(pdgpu_batch *b, int32_t system, double *xyz, size_t stride_bytes);
int pdgpu_batch_set_velocities(pdgpu_batch *b, int32_t system, const double *xyz, size_t stride_bytes);
/* Forces of all systems (concatenated atoms, AoS, J/m, ADDED to f_accum, may be
 * NULL) and per-system energies (energies[n_systems], may be NULL). */
int pdgpu_batch_compute(pdgpu_batch *b, uint32_t components, double *f_accum, pdgpu_energies *energies);
/* n_steps MD steps of every system as one hipGraph-replayed device step.  Traces
 * (may be NULL) receive n_steps * n_systems values, step-major (J). */
int pdgpu_batch_md(pdgpu_batch *b, const pdgpu_md_params *p, int32_t n_steps, double *epot_trace,
                   double *ekin_trace);
/* REX_Local::runcore (remd.cpp:65-254): n_rounds of {every replica runs
 * p->total_steps steps; alternating even/odd neighbour exchanges with
 * exchangeCriterion (remd.cpp:349-357)}.  System s is the replica at the s-th
 * temperature; accepted structures swap between neighbours with velocities
 * rescaled by sqrt(T ratio).  accepted/attempted count exchanges per pair
 * (s, s+1); final_epot gets the last round's replica energies (J).  The
 * Metropolis uniforms come from Philox4x32-10 keyed by `seed`. */
int pdgpu_batch_remd(pdgpu_batch *b, const pdgpu_md_params *p, int32_t n_rounds, uint64_t seed,
                     int32_t *accepted, int32_t *attempted, double *final_epot);

/* ---- instrumentation ---------------------------------------------------------------- */

/* Kernel timing (no counterpart in PD, whose MD timer has 1 s resolution,
 * md.cpp:194-196).  enable = k >= 1 brackets every k-th launch of each named
 * kernel ("nonbonded", "prune", "pair_search", "gb_radii", "gb_pair", "gb_chain",
 * "lcpo"; "list_build" spans a whole list rebuild, cleanSpace to the pair search) with HIP events on the engine's own stream; enable = 0 turns timing off.
 * Each event pair costs the queue a few microseconds, so a sampling interval keeps
 * long runs close to their untimed speed.  Enabling resets the totals. */
int pdgpu_set_timing(pdgpu_engine *e, int32_t enable);
/* Summed duration (ms) and launch count of one named kernel since timing was enabled. */
int pdgpu_kernel_time(pdgpu_engine *e, const char *kernel, double *total_ms, int64_t *launches);

#ifdef __cplusplus
}
#endif
#endif
