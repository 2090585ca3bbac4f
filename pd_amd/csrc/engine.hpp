// engine.hpp -- internal state of one pdgpu engine (one molecular system in HBM).
//
// Layout in HBM (all device buffers are owned by Engine):
//   original order (PD atom index):  x,y,z,vx,vy,vz (f64 SoA), mass (f64),
//       bonded+GB force accumulators fbx,fby,fbz (int64 fixed point, 2^32 per
//       kcal/mol/A), molecules (first,last), bond-order band/sparse tables.
//   cluster order (rebuilt with the list): slots of 8 atoms per cluster, atoms
//       of a cluster taken from one grid column sorted by z.  slot_orig[slot]
//       maps back to the PD index (-1 for padding); spos (f64 x,y,z + pad, 32 B)
//       holds the positions gathered each step (spos32: the same in f32, 16 B,
//       for the prune), sprm (f32 scaled charge, LJ
//       radius, sqrt(eps), 16 B) the pair parameters; nbx,nby,nbz (int64) the nonbonded force
//       accumulators in slot order.  Work groups of up to 4 clusters of one
//       column share a candidate j-cluster table (wg_cand).
//   list: for every i-cluster a contiguous run of 8-byte entries
//       {j slot | image<<24 | j-has-LJ<<29 ; listed-mask(8) | bond-order codes(16)
//       | candidate rank<<24} (see k_list.hip), located by cl_entry_start /
//       cl_entry_count.  The pruned copy (pentries) keeps the entries whose j atom
//       has an LJ epsilon from the front of each cluster's run (pcount of them)
//       and the others from the back (pcount_nolj, last one first).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <map>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/pdgpu.h"

namespace pdgpu {

// Fixed-point scale of all force / energy-derivative accumulators: 2^32 units
// per kcal/mol/A.  |F| up to 2^31 kcal/mol/A fits an int64.
constexpr double kFixScale = 4294967296.0;
constexpr float kFixScaleF = 4294967296.0f;
constexpr int kClusterSize = 8;
// Nonbonded work groups: up to kGroup consecutive i-clusters of one grid column,
// one wavefront each.  Their list shares one table of up to kGroupRanks
// candidate j-clusters, which the nonbonded kernel mirrors in LDS to sum the j
// forces before touching global memory (rank kGroupRanks = no LDS slot).
// 127 ranks keep the table at 24 KB of LDS, so four work groups share a CU; the
// rarer j-clusters beyond it add straight to global memory.
constexpr int kGroup = 4;
constexpr int kGroupRanks = 127;
constexpr int kGroupStride = 128;
constexpr int kWave = 64;

// PD constants (forcefield.cpp:35-55), FP64.
struct Consts {
  static constexpr double PI = 3.14159265358979323846;
  static constexpr double kcal2J = 4184.0;
  static constexpr double Na = 6.0221418E23;
  static constexpr double kB = 1.38065E-23;
  static constexpr double Angstrom = 1E-10;
  static constexpr double e_charge = 1.60217645E-19;
  static constexpr double e0 = 8.854187817E-12;
  static constexpr double Bar2Pa = 100000.0;
  static double J2kcal() { return 1.0 / kcal2J; }
  static double four_pi_e0() { return (PI * 4.0) * e0; }
  static double econv() {  // kcal/mol * A
    return (J2kcal() * Na * (e_charge * e_charge)) / (four_pi_e0() * Angstrom);
  }
  static double halfeconv() { return econv() * 0.5; }
  static double econv_joule() { return (e_charge * e_charge) / (four_pi_e0() * Angstrom); }
  static double halfeconv_joule() { return econv_joule() * 0.5; }
  // kcal/mol -> J per molecule; kcal/mol/A -> J/m
  static double kcal_to_J() { return kcal2J / Na; }
  static double J_to_kcalmol() { return J2kcal() * Na; }
  static double kcalA_to_Jm() { return kcal2J / Na / Angstrom; }
};

struct EngineError : std::runtime_error {
  int code;
  EngineError(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

#define PDGPU_HIP(call)                                                                  \
  do {                                                                                   \
    hipError_t _e = (call);                                                              \
    if (_e != hipSuccess)                                                                \
      throw ::pdgpu::EngineError(PDGPU_ERR_HIP, std::string(#call) + ": " +              \
                                                    hipGetErrorString(_e));              \
  } while (0)

template <typename T>
struct DBuf {
  T *p = nullptr;
  size_t n = 0;
  DBuf() = default;
  DBuf(const DBuf &) = delete;
  DBuf &operator=(const DBuf &) = delete;
  ~DBuf() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  void resize(size_t count) {  // contents are not preserved
    if (count <= n && p) return;
    release();
    size_t bytes = (count ? count : 1) * sizeof(T);
    if (hipMalloc(&p, bytes) != hipSuccess)
      throw EngineError(PDGPU_ERR_NOMEM, "device allocation of " + std::to_string(bytes) + " bytes failed");
    n = count;
  }
  void upload(const T *h, size_t count, hipStream_t s) {
    resize(count);
    if (count) PDGPU_HIP(hipMemcpyAsync(p, h, count * sizeof(T), hipMemcpyHostToDevice, s));
  }
  void upload(const std::vector<T> &h, hipStream_t s) { upload(h.data(), h.size(), s); }
  void download(T *h, size_t count, hipStream_t s) const {
    if (count) PDGPU_HIP(hipMemcpyAsync(h, p, count * sizeof(T), hipMemcpyDeviceToHost, s));
  }
};

// Host memory the GPU reads and writes directly (pinned), grown as needed: results
// and states cross the bus in one kernel's loads or stores, where a copy to or from
// pageable memory goes through the runtime's own staging.
struct HostStage {
  double *p = nullptr;
  size_t n = 0;
  HostStage() = default;
  HostStage(const HostStage &) = delete;
  HostStage &operator=(const HostStage &) = delete;
  ~HostStage() {
    if (p) (void)hipHostFree(p);
  }
  double *need(size_t count) {
    if (count > n) {
      if (p) (void)hipHostFree(p);
      p = nullptr;
      n = 0;
      if (hipHostMalloc(reinterpret_cast<void **>(&p), count * sizeof(double)) != hipSuccess) {
        (void)hipGetLastError();
        p = nullptr;
        throw EngineError(PDGPU_ERR_NOMEM,
                          "pinned host allocation of " + std::to_string(count * sizeof(double)) + " bytes failed");
      }
      n = count;
    }
    return p;
  }
};
// xyz vectors between the caller's array (any stride) and device SoA arrays; both
// return when the data have arrived (state_io.hip)
void xyz_to_device(HostStage &st, hipStream_t s, const double *xyz, size_t stride_bytes, int n, double *x, double *y,
                   double *z);
constexpr int kStagePiece = 1 << 18;  // atoms in pinned memory at once (6 MiB)
void xyz_to_host(HostStage &st, hipStream_t s, const double *x, const double *y, const double *z, int n, double *xyz,
                 size_t stride_bytes);

// A trace of `count` doubles on its way to the caller: pinned up to 8 MiB, else pageable.
struct TraceFetch {
  std::vector<double> big;
  const double *get(HostStage &st, const DBuf<double> &d, size_t count, hipStream_t s) {
    double *h;
    if (count <= (size_t)1 << 20) {
      h = st.need(count);
    } else {
      big.resize(count);
      h = big.data();
    }
    d.download(h, count, s);
    PDGPU_HIP(hipStreamSynchronize(s));
    return h;
  }
};

// Position of one cluster slot: one 32-byte record, so a lane fetches it with
// two 16-byte loads.
struct alignas(32) SlotPos {
  double x, y, z, pad;
};

// Parameters the nonbonded kernel needs, in the kernel's units (kcal/mol, A).
// The FP32 constants of NBKernelParams that the FP64 pair arithmetic takes, unrounded.
struct NBFine {
  double vdw14, elec14, vdwinner, invw_vdw, invw2_vdw4, inner, invw_el, invw2_el4;
  double fcut, eshift, fs_c1, fs_c2, fs_c3, fs_c4, fs_invw, fs_x0;
};
struct NBKernelParams {
  double cut2;        // Cutoff^2 (FP64: PD's per-pair test, nonbonded.cpp:720)
  double vdwcut2;     // VdwCutoff^2
  double vdwcut_d;    // VdwCutoff: PD's LJ test is on the distance (nonbonded.cpp:742)
  float cut, inner, vdwcut, vdwinner;
  float invw2_vdw4;   // 4 / (VdwCutoff-VdwInnerCutoff)^2
  float invw_vdw;
  float invw_el, invw2_el4;
  float sA, sB, sC, sD, sE, fcut, eshift;  // force-switch constants (nonbonded.cpp:620-636)
  float rc2, rin2;
  float fs_c1, fs_c2, fs_c3, fs_c4;  // sA*sB, sA*sC, sA*sD, sA*sE: the outer energy in Horner form
  float fs_k;                        // rc2 - 3 rin2
  float fs_invw, fs_x0;              // 1 / (rc2 - rin2) and -rin2 / (rc2 - rin2) (0 without a switch region)
  int same_cut;                      // Cutoff == VdwCutoff: one cutoff test per pair
  float vdw14, elec14;
  int vdw_on;
  int elec_mode;      // 0 none, 1 plain, 3 energy switch, 4 force switch
  double vdwcor_per_atom;  // kcal/mol added per atom when VdwCor
  bool fine;               // FP64 pair arithmetic (set per launch), with
  NBFine d;
};

// ---- Generalized Born (k_gb.hip) ------------------------------------------------
// Kernel constants of FF_GeneralizedBorn_Still in kcal/mol and A.
struct GBK {
  double cut2;          // Cutoff^2
  double cut;           // Cutoff
  double still2;        // GbsaStillCutoff^2
  double vdw_lim;       // sqrt(r2) < VdwCutoff is r2 < vdw_lim (gbff.cpp:1686)
  double gb_lim;        // sqrt(r2) <= Cutoff is r2 < gb_lim (gbff.cpp:560)
  double premul_d;      // -halfeconv (1/eps_in - 1/eps_out), kcal/mol A
  double ec_in_d;       // econv / eps_in
  float premul2;        // 2 premul_d
  float ec_in, ec_out, ec_ratio;  // ec_in_d, econv / eps_out, eps_in / eps_out
  float inner, invw, invw2_4;
  float vdwinner, vinvw, vinvw2_4;
  float thresh;         // ExpApproxThreshold
  float P4, invP5, half_pi_P5;  // P4, 1 / P5, pi P5 / 2
  float vdw14, elec14;
  float inside, outside, far_k, fix_lim, edge;  // per pass (GBState::set_params)
};
// A piece of work of the GB passes: i tiles ti .. ti+ni-1 (ni 1 or 2) against j
// tiles tj .. tj+nj-1 (indices over all systems' tiles), the table of its pair codes
// (-1: none), its energy slot (contiguous within a system).
struct GBTask {
  int sys, ti, ni, tj, nj, code, slot, pad;
};
// A tile's centre, the largest distance of an atom from it, its largest GB radius
// and its largest Born radius, at the current positions.
struct GBTile {
  double x, y, z, rad;
  float rmax, amax;
};
struct GBPassArgs {
  GBK K;
  const GBTask *tasks;
  const int2 *tile_atoms;  // per tile: first atom, atoms
  const GBTile *tiles;
  const unsigned *codes;
  const double *x, *y, *z;
  const float *q, *ljr, *lje, *bornf, *gbrad, *Vj;
  const double *born;
  const long long *deda_in;
  long long *s0, *s1, *s2, *s3;  // the pass's sums per atom
  double *e_part;
};
struct GBSys {
  int first, count;     // atom range in the concatenated arrays
  int mid;              // BondOrder::m_MaxIndexDelta
  long band_off;        // offset of the system's band matrix in the concatenated array
  int sp_base;          // offset of the system's sparse CSR offsets (count+1 entries)
};

struct Engine;
// The per-step trace entry of pdgpu_md, written after the step's energy sums.
struct StepRecord {
  double *trace;
  int step;
  int use_nb, use_bonded, use_gb, use_sasa;
  double vdwcor, kcal_to_J;
};

constexpr int kMaxSums = 8;
constexpr int kSumThreads = 256;
struct SumList {
  const double *part[kMaxSums];
  double *out[kMaxSums];
  int count[kMaxSums];
  int n;
  int record;
  StepRecord rec;
  const double *e_out;
};

// Device pointers of FF_Bonded terms (k_bonded.hip); force constants in kcal/mol units.
struct BondedArrays {
  int nb, na, nt;
  const int *bi, *bj;
  const double *bl, *bk;
  const int *ai, *aa, *aj;
  const double *at0, *ak;
  const int *ti, *ta, *tb, *tj, *tterms;
  const double *tvn, *tnn, *tgamma;
  const int2 *win;  // per block: first atom of its LDS force window and the window length (0: direct)
};
// Blocks of 256 terms never mix bonds, angles and torsions; a block whose terms
// touch at most kBondedWindow consecutive atoms sums its forces in LDS first.
// The window is the size of the nonbonded kernel's j-force table, whose LDS the
// bonded workgroups of that kernel use.
constexpr int kBondedWindow = kGroupRanks * kClusterSize;
int bonded_blocks(int nb, int na, int nt);
std::vector<int2> bonded_windows(int nb, const int *bi, const int *bj, int na, const int *ai, const int *aa,
                                 const int *aj, int nt, const int *ti, const int *ta, const int *tb, const int *tj);
void launch_bonded_kernel(hipStream_t s, const BondedArrays &B, const double *x, const double *y,
                          const double *z, long long *fx, long long *fy, long long *fz, double *partial,
                          double *eterm);

// Device arrays of the GB passes for one or more systems laid end to end.
// GB energy slots (kcal/mol: cross, vdw, elec, -, self) added to PD's terms (J);
// pol_terms false: the polarisation energy goes into epot only (FastMode off).
void gb_slots_to_energies(const double *h, bool pol_terms, pdgpu_energies &e);

// Constants of the plain GB comparator (k_gb.hip), FP64, kcal/mol and A.
struct PlainGB {
  int n, mid;
  double still2, cut2, vdwcut, inner, vdwinner, invw, vinvw, premul, ec_in, ec_out, thresh;
  double P4, P5, invP5, vdw14, elec14, halfeconv, offset, pi;
};
// What shares the opening launch of a GB evaluation (k_gb_open): the bonded terms, whose
// 256-term blocks have no matrix of pairs to hide behind, and a previous step's sums.
struct GBOpen {
  BondedArrays bonded;
  int bonded_blocks = 0;
  double *bonded_partial = nullptr, *bonded_eterm = nullptr;
  const struct SumList *sums = nullptr;
};
// The final energy sums of a GB evaluation, for a launch that other sums share
// (gb_sums_block): per system the tile pairs' and the self energies.
struct GBSums {
  const double *part, *eself;
  const int *beg, *end, *first, *count;
  double *out;
  int stride, off;
  int slots;  // of the tile pairs' four sums written (the fourth is zero)
};
struct GBState {
  pdgpu_gb_params prm{};
  GBK kp{}, kr{};  // of the pair pass; of radii and chain
  int n_atoms_total = 0;
  std::vector<GBTask> h_tasks;
  std::vector<GBSys> h_sys;
  std::vector<int2> h_tile_atoms;
  std::vector<std::vector<std::pair<int, int>>> h_linked;  // per system: tile pairs with a sparse partner
  std::vector<int8_t> h_band;
  std::vector<int> h_sp_off, h_sp_part, h_sp_ord, h_tile_beg, h_slot_beg, h_slot_end, h_coded;
  int n_slots = 0;
  DBuf<GBTask> tasks;
  DBuf<GBSys> sysd;
  DBuf<int2> tile_atoms;
  DBuf<GBTile> tiles;
  DBuf<unsigned> codes;
  DBuf<int8_t> band;
  DBuf<int> sp_off, sp_part, sp_ord, slot_beg, slot_end, sys_first, sys_count, coded;
  DBuf<long long> gpol, deda;
  DBuf<double> born, eself, e_part, terms123;
  DBuf<float> bornf, q, ljr, lje, gbrad, Vj;
  ~GBState();
  void set_params(const pdgpu_gb_params &p);
  void add_system(int first, int count, int mid, const std::vector<int8_t> &band_sys, const std::vector<int> &spi,
                  const std::vector<int> &spj, const std::vector<int> &spo);
  void upload(hipStream_t s);
  void run(hipStream_t s, const double *x, const double *y, const double *z, long long *fx, long long *fy,
           long long *fz, double *out, int out_stride, int out_off, Engine *timer_owner, bool energy_only = false,
           const GBOpen *open = nullptr, bool sums = true);  // sums = false: left to the caller (sum_args)
  GBSums sum_args(double *out, int out_stride, int out_off, int slots = 4) const {
    return GBSums{e_part.p, eself.p, slot_beg.p, slot_end.p, sys_first.p, sys_count.p, out, out_stride, out_off, slots};
  }
  // wavefronts per task of the radii, pair and chain passes (1, 2 or 4; 0: by the
  // number of tasks)
  int split[3] = {0, 0, 0};
  void make_tasks();
  GBPassArgs pass_args(const double *x, const double *y, const double *z, long long *fx, long long *fy,
                       long long *fz) const;
  template <int PASS>
  void launch_pass(hipStream_t s, const GBPassArgs &A, int sp);
  // the plain comparator (one thread per atom, FP64 sums): on for a single system
  bool plain = false;
  DBuf<double> pl_q, pl_r, pl_e, pl_gr, pl_vj, pl_deda, pl_e3;
  PlainGB plain_args() const;
  void set_split(const int32_t *s3);
  // times each tile kernel at every split on the current positions and keeps the
  // fastest; us[3*k + m] = average launch (us) of kernel k at split 1 << m
  void autotune(hipStream_t s, const double *x, const double *y, const double *z, long long *fx, long long *fy,
                long long *fz, double *out, int out_stride, int out_off, double *us);
};

// ---- LCPO SASA (k_lcpo.hip) ------------------------------------------------------
constexpr int kLcpoMax = 80;  // Nlistmax, lcpo.h:24
struct LCPOState {
  int n = 0;
  int update = 5;  // FF_SASA_LCPO::UpdateSasa (lcpo.h:67)
  std::vector<int8_t> h_use;
  std::vector<double> h_R, h_P, h_sig;  // radius + 1.4 A, P1..P4, sigma (J/A^2 per molecule)
  std::vector<int> h_atom_sys, h_first, h_count;
  DBuf<int8_t> use;
  DBuf<double> R, sig, nl_s, sasa, dvx, dvy, dvz, eatom;
  DBuf<double4> P, pr;  // P1..P4; packed position + radius (R < 0: not used)
  DBuf<double> tile_box;  // box of each 64-atom tile's used atoms (lo xyz, hi xyz)
  double max_R = 0.0;
  DBuf<int> atom_sys, sys_first, sys_count, nl_cnt, nl_idx;
  void add_system(int first, int count, const int8_t *use, const double *radius, const double *P4,
                  const double *sigma_j);
  void append(const LCPOState &o, int first);  // another system's atoms, as they are
  void upload(hipStream_t s);
  // full: recompute now; otherwise recompute when step % update == 0 and re-apply
  // the stored forces otherwise.  block_part: the energies' 4-wide block sums too;
  // gb: the launch of the forces also takes these energy sums
  void run(hipStream_t s, const double *x, const double *y, const double *z, long long *fx, long long *fy,
           long long *fz, int step, bool full, bool energy_only = false, double *block_part = nullptr,
           const GBSums *gb = nullptr);
  // a step that takes the stored areas and forces again
  bool reapplies(int step) const { return update > 0 && step % update != 0; }
};

void gb_fixed_terms(int n, const double *gbrad, const pdgpu_gb_params &p, const int32_t *off12,
                    const int32_t *idx12, const double *d12, const int32_t *off13, const int32_t *idx13,
                    const double *d13, std::vector<double> &Vj, std::vector<double> &terms123);

struct Engine {
  int n = 0;
  int device = 0;
  hipStream_t stream = nullptr;
  std::string last_error;

  // ---- system description -------------------------------------------------
  std::vector<double> h_radius, h_epsilon, h_charge, h_mass;
  std::vector<int> h_mol_first, h_mol_last;
  int mid = 1;                 // BondOrder::m_MaxIndexDelta
  std::vector<int8_t> h_band;  // mid*(n-1)
  std::vector<int> h_sp_i, h_sp_j, h_sp_order;
  bool periodic = false;
  double box[3] = {0, 0, 0};
  double last_pressure = 0.0;  // Bar, of the last barostat step
  double list_cutoff = 0.0;    // NeighbourListBase::Cutoff
  double padding = 0.5;        // NeighbourListBase::Padding default (neighbourlist.cpp:35)
  bool calc_shadow = false;
  uint32_t full_update_count = 0;
  bool have_nb = false;
  pdgpu_nb_params nb{};
  NBKernelParams nbk{};
  bool have_positions = false;
  bool list_valid = false;

  // ---- device state, original order -----------------------------------------
  DBuf<double> x, y, z, vx, vy, vz, mass;
  DBuf<double> fox, foy, foz;  // Beeman's old forces (J/m), PD's oldatom[i].f
  DBuf<double> thermo;         // [0] Berendsen's chi of the step
  DBuf<double> mom_part, mom;  // momentum-step partials and totals
  void remove_momentum();      // run_core's momentum step with a thermostat
  DBuf<long long> fbx, fby, fbz;           // bonded / GB / integrator force accumulators
  DBuf<int> mol_first, mol_last;
  DBuf<int8_t> band;
  DBuf<int> sp_off, sp_part, sp_ord;       // per-atom CSR of off-diagonal partners (both directions)
  DBuf<float> q_scaled, lj_r, lj_e;        // per atom, original order
  DBuf<float4> prm_lo;                     // what FP32 leaves of the three

  // ---- cluster / list state ---------------------------------------------------
  int ncx = 0, ncy = 0, ncol = 0;
  double grid_lo[3] = {0, 0, 0}, grid_w[2] = {0, 0};
  int max_clusters = 0;                    // allocation bound
  DBuf<double> wx, wy, wz;                 // wrapped coordinates used for binning
  DBuf<int> atom_wrap;                     // binning wrap counts, one byte per axis
  DBuf<unsigned char> slot_list;           // per-slot pair-search records (k_list.hip)
  DBuf<int> atom_col, col_count, col_fill, col_atom_start, col_cl_start, col_ncl;
  DBuf<int> col_atoms;                     // atoms grouped by column (unsorted)
  DBuf<int> slot_orig, orig_slot;
  DBuf<int> n_clusters_d;                  // device scalar
  DBuf<int> cl_col;                        // column of each cluster
  DBuf<double> cl_lo, cl_hi;               // cluster bounding boxes (wrapped frame), 3 per cluster
  DBuf<SlotPos> spos;                      // gathered FP64 positions, slot order
  DBuf<float4> spos32;                     // the same positions in FP32 (x, y, z, 0) for the prune
  DBuf<float4> sprm;                       // per slot: scaled charge, LJ radius, sqrt(eps), 0
  DBuf<float4> sprm_lo;                    // the FP64 values less those (prm_lo by slot)
  int max_groups = 0;                      // allocation bound of work groups
  DBuf<int> col_grp_start, grp_first, grp_count, n_groups_d;
  DBuf<int> grp_order, grp_work;           // the nonbonded kernel's block -> group map (8 * nb_per_cap blocks)
  int nb_per_cap = 0;
  int nb_parts = 1, nb_share = 1;          // nonbonded kernel: workgroups per group, and waves per cluster in each
  bool order_due = false;                  // the next prune launch computes grp_order (set by a list build)
  DBuf<int> wg_ncand, wg_cand;             // per group: candidate j-cluster table (kGroupStride each)
  DBuf<long long> nbx, nby, nbz;           // nonbonded force accumulators, slot order
  DBuf<uint2> entries;
  DBuf<int> cl_entry_start, cl_entry_count;
  // pruned copy of the list: the entries with a pair within Cutoff + prune_margin
  // at the prune positions pref; valid while every atom stays within
  // prune_margin / 2 of pref (checked on the device each step)
  DBuf<uint2> pentries;
  DBuf<int> pcount, pcount_nolj;
  DBuf<SlotPos> pref;
  DBuf<unsigned> prune_dmax;               // max displacement from pref (float bits): 2 alternating sets of spread words
  int dmax_cur = 0;                        // which prune_dmax word this evaluation fills
  // 0.4 A: on the 98,304-atom NVE water box 0.35 / 0.4 / 0.5 / 0.6 / 0.7 A gave
  // 405.7 / 407.5 / 402 / 403.3 / 396.2 ns/day (a larger margin prunes less
  // often but leaves more entries to the force kernel)
  double prune_margin = 0.4;
  bool prune_forced = true;
  DBuf<unsigned long long> entry_counter;  // [0] entries used, [1] overflow flag
  size_t entry_capacity = 0;
  int n_clusters = 0;                      // host copy after a build
  // The rebuild inside pdgpu_md reads its counters back into pinned memory
  // without waiting; the step checks them once its force kernels are queued.
  unsigned long long *h_list_check = nullptr;  // [0] entries, [1] overflow, [2] candidate overflow, [3] clusters
  hipEvent_t list_event = nullptr;
  bool list_check_pending = false;
  bool finish_list_check();                // false: the list overflowed (room already grown)
  bool grow_list_room();                   // after a search: grow passes / capacity; false if it all fitted
  static constexpr int kMaxListPasses = 64;
  int list_passes = 1;                     // pair-search passes over disjoint shares of the stencil

  // ---- reductions ---------------------------------------------------------------
  DBuf<double> e_partial;                  // per-workgroup nonbonded energy partials (4 per group and part)
  DBuf<double> e_partial_b;                // the alternate array: consecutive evaluations switch
  int e_partial_sel = 0;
  SumList nb_sums{};                       // a previous MD step's sums, run by the nonbonded kernel
  bool nb_sums_pending = false;
  DBuf<double> e_partial_bonded;           // per-block bonded energy partials (4 per block)
  DBuf<double> e_partial_ke;               // per-block kinetic energy partials (4 per block)
  DBuf<double> e_out;                      // reduced energies, 4 per component (see Slots)
  DBuf<double> trace;                      // per-step epot / ekin of pdgpu_md
  // energy partials (4 per block) summed by one kernel at the end of an
  // evaluation, or of an MD step together with its trace entry
  struct PendingSum {
    const double *part;
    int count;
    double *out;
  };
  std::vector<PendingSum> pending_sums;
  void defer_sum4(const double *part, int count, double *out) { pending_sums.push_back({part, count, out}); }
  void flush_sums(const StepRecord *rec = nullptr);
  // pdgpu_md: a step's sums (at most kMaxSums lists) wait for the next step's
  // opening kernel, which runs them in its first workgroup
  SumList fused_sums{};
  bool fused_pending = false;
  void run_fused_sums();  // the deferred sums in a launch of their own
  void defer_step_sums(const StepRecord &rec);

  // ---- bonded terms -------------------------------------------------------------
  int nbonds = 0, nangles = 0, ntors = 0;
  DBuf<int> b_i, b_j, a_i, a_a, a_j, t_i, t_a, t_b, t_j, t_terms;
  DBuf<int2> b_win;
  DBuf<double> b_l, b_k, a_t0, a_k, t_vn, t_nn, t_gamma;

  explicit Engine(int natoms, int dev);
  ~Engine();

  void require(bool cond, const char *msg) const {
    if (!cond) throw EngineError(PDGPU_ERR_ARG, msg);
  }
  void sync() { PDGPU_HIP(hipStreamSynchronize(stream)); }

  // list.hip
  void build_list(bool deferred = false);  // deferred: the overflow check waits for finish_list_check
  // export.hip: the list in PD's packed form
  int64_t count_pairs();
  void export_pairs(int32_t *counts, uint32_t *packed, int64_t capacity);
  DBuf<int> ex_count;
  DBuf<unsigned long long> ex_start, ex_total;
  DBuf<uint32_t> ex_packed;
  // kernel timing instrumentation (HIP events on `stream`)
  bool timing = false;
  struct TimerSlot {
    double ms = 0.0;
    long long launches = 0;  // launches timed
    long long calls = 0;     // launches seen while timing was on
    std::vector<std::pair<hipEvent_t, hipEvent_t>> pending;
  };
  int timing_every = 1;  // time every k-th launch of each named kernel
  bool timer_sample(const char *name) {
    if (!timing) return false;
    return (timers[name].calls++ % timing_every) == 0;
  }
  std::map<std::string, TimerSlot> timers;
  std::vector<hipEvent_t> event_pool;
  hipEvent_t take_event();
  void resolve_timers();
  // nonbonded.hip
  void prepare_slots();
  void setup_nonbonded(const pdgpu_nb_params &p);
  // energies: vdw, elec, virial; partial: the per-workgroup energy partials
  // (max_groups * nb_parts * 4 doubles), by default the engine's own e_partial
  // bonded_slots: the bonded terms run in the same launch (their sums go there)
  void launch_nonbonded(double *energy_slots, bool forces = true, double *partial = nullptr,
                        double *bonded_slots = nullptr);
  void size_eval_buffers();  // every buffer an evaluation writes, sized at a list build
  // bonded.hip
  // energies: bond, angle, torsion, virial; partial: bonded_blocks * 4 doubles
  void launch_bonded(double *energy_slots, double *partial = nullptr);
  BondedArrays bonded_arrays() const;
  // integrate.hip
  // clears accumulators and the energy slots eo (default e_out) and gathers slot positions
  // opened: the previous MD step's integrator did the opening kernel's work
  // (running it anyway would be harmless: the same values again)
  // gb_next: without the nonbonded term, the pending sums are left to the GB opening
  void begin_evaluation(bool nonbonded, double *eo = nullptr, bool opened = false, bool gb_next = false);
  void forces_to_host(double *f, size_t stride_bytes);
  HostStage stage;    // states, forces and traces on their way to or from the host
  // forces + energies into e_out (step < 0: LCPO in full); flush = false leaves the
  // energy sums pending for the caller's flush_sums
  void evaluate(uint32_t components, int step = -1, bool flush = true);
  void energies_to_host(uint32_t components, pdgpu_energies *out);
  void energies_from_slots(uint32_t components, const double *h, pdgpu_energies *out) const;
  // noalloc.hip: the allocation-free evaluation of pdgpu_compute_noalloc
  double *scratch = nullptr;               // this device's file-scope scratch array (device address)
  double *h_eout = nullptr;                // pinned: the energy slots, a partial update's results
  void evaluate_noalloc(uint32_t components, double *d_f, size_t stride_bytes, pdgpu_energies *out);
  // times trial_steps MD steps at each prune margin from the same state and keeps
  // the fastest (the state is restored; the next evaluation rebuilds the list)
  double autotune_md(const pdgpu_md_params &p, int trial_steps, int n_margins, const double *margins, bool retune,
                     double *ms);
  // open_next: the integrator also does the next step's opening work (that step
  // keeps the list, no thermostat or barostat); its begin_evaluation launches nothing
  void integrate(const pdgpu_md_params &p, int step, double *ekin_slot, bool open_next = false);
  bool opened_ahead = false;
  // k_protocols.hip
  DBuf<double> ox, oy, oz;  // the minimiser's last accepted positions (PD's old snapshot)
  DBuf<double> sd_state;    // reference energy (J), step multiplier, decision
  void minimise(const pdgpu_min_params &p, int n_steps, double *epot_trace);
  // FF_NonBonded::calcEnergies with UsePartialRecalc (k_partial.hip): the
  // positions and energy terms (J) of the last evaluation, and the list's
  // full-update count then
  DBuf<double> pr_x, pr_y, pr_z, pr_part, pr_rad, pr_eps, pr_chg;
  DBuf<int> pr_moved;
  bool pr_valid = false;
  uint32_t pr_update_count = 0;
  double pr_vdw = 0.0, pr_elec = 0.0;
  void energy_update(uint32_t components, pdgpu_energies *out);
  void initial_speeds(double temperature, uint64_t seed, uint32_t noise_stream);
  void md(const pdgpu_md_params &p, int n_steps, double *epot_trace, double *ekin_trace);
  // trajectory frames of the last md call (UpdateTra): positions (SoA per frame)
  // and the step's energy slots, kept on the device until read
  DBuf<double> frame_xyz, frame_e;
  std::vector<int> h_frame_steps;
  uint32_t frame_components = 0;
  void get_frames(int max_frames, double *xyz, int32_t *steps, pdgpu_energies *energies, int32_t *n_frames);
  void write_snapshot(const char *path, const char *name, bool append);
  void read_snapshot(const char *path, const char *name);
  uint32_t last_components = 0;
  // k_lcpo.hip
  std::unique_ptr<LCPOState> lcpo;
  DBuf<double> e_partial_lcpo;
  // with_gb: the launch of the surface energies also runs the GB energy sums
  void launch_lcpo(double *energy_slot, int step, bool full, bool energy_only = false, const GBSums *with_gb = nullptr);
  // k_gb.hip
  bool have_gb = false;
  std::unique_ptr<GBState> gb;
  // bonded_slots: the bonded terms run in the opening launch (their sums go there)
  void launch_gb(double *energy_slots, bool energy_only = false, double *bonded_slots = nullptr, bool sums = true);
  SumList gb_sums{};  // a previous step's sums, for that launch
  int gb_bonded_sel = 0;

};

// Brackets the launches in its scope with HIP events on the engine's stream
// when timing is on (pdgpu_set_timing).
struct ScopedTimer {
  Engine &E;
  const char *name;
  bool on;
  hipEvent_t a = nullptr, b = nullptr;
  ScopedTimer(Engine &e, const char *n) : E(e), name(n), on(e.timer_sample(n)) {
    if (on) {
      a = E.take_event();
      (void)hipEventRecord(a, E.stream);
    }
  }
  ~ScopedTimer() {
    if (on) {
      b = E.take_event();
      (void)hipEventRecord(b, E.stream);
      auto &slot = E.timers[name];
      slot.pending.emplace_back(a, b);
      if (slot.pending.size() > 4096) E.resolve_timers();
    }
  }
};

// ScopedTimer for code paths that may run without an owning Engine.
struct ScopedTimerOpt {
  Engine *E;
  const char *name;
  bool on;
  hipEvent_t a = nullptr;
  ScopedTimerOpt(Engine *e, const char *n) : E(e), name(n), on(e && e->timer_sample(n)) {
    if (on) {
      a = E->take_event();
      (void)hipEventRecord(a, E->stream);
    }
  }
  ~ScopedTimerOpt() {
    if (on) {
      hipEvent_t b = E->take_event();
      (void)hipEventRecord(b, E->stream);
      E->timers[name].pending.emplace_back(a, b);
    }
  }
};

void langevin_coefficients(double gammat, double *c6);
// noalloc.hip: device address of `device`'s scratch array, looked up once per device
double *scratch_for_device(int device);


// ---- device helpers ------------------------------------------------------------

// floor(v * 2^32) as a 64-bit integer, exactly: d = v * 2^32 is exact, hi is its
// upper 32 bits (floor), lo = d - hi * 2^32 lies in [0, 2^32) and is exact, so
// two 32-bit conversions build the result (|v| < 2^31 kcal/mol/A).
__device__ __forceinline__ long long fix_from_double(double v) {
  const double d = v * kFixScale;
  const double hi = floor(d * (1.0 / kFixScale));
  const double lo = fma(hi, -kFixScale, d);
  const unsigned long long h = (unsigned long long)(unsigned)(int)hi;
  return (long long)((h << 32) | (unsigned long long)(unsigned)lo);
}
// The same value for an FP32 input in one step fewer: floor(v * 2^32) / 2^32 =
// floor(v), and v - floor(v) is exact in FP64, so lo = (v - floor(v)) * 2^32.
__device__ __forceinline__ long long fix_from_float(float v) {
  const double d = (double)v;
  const double hi = floor(d);
  const double lo = (d - hi) * kFixScale;
  const unsigned long long h = (unsigned long long)(unsigned)(int)hi;
  return (long long)((h << 32) | (unsigned long long)(unsigned)lo);
}
__device__ __forceinline__ void fix_add(long long *p, long long v) {
  atomicAdd(reinterpret_cast<unsigned long long *>(p), static_cast<unsigned long long>(v));
}

// Philox4x32-10 (Salmon, Moraes, Dror & Shaw, SC'11): the counter-based
// generator behind every random stream of the engine.
__device__ __forceinline__ void philox_round10(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; r++) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
    const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
    const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
    const uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
    c[0] = n0;
    c[1] = lo1;
    c[2] = n2;
    c[3] = lo0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

// A uniform double in (0, 1] from two 32-bit words (53 bits).
__device__ __forceinline__ double uniform53(uint32_t a, uint32_t b) {
  const uint64_t m = ((uint64_t)(a >> 5) << 26) | (uint64_t)(b >> 6);
  return ((double)m + 1.0) * (1.0 / 9007199254740992.0);
}

// The wave's butterfly without LDS: the partners 32 and 16 lanes away come from the
// lane swaps, those 8, 4, 2 and 1 away from DPP operands (a rotation of the 16-lane row
// by 8; by 4, once lanes 8 apart agree; a quad's permutations).  A swap of a value with
// itself leaves both partners' values in each of the two lanes.  __shfl_xor goes
// through the LDS crossbar: six dependent trips of ~100 cycles for each word.
template <int CTRL>
__device__ __forceinline__ unsigned dpp_word(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
constexpr int kRowRor8 = 0x128, kRowRor4 = 0x124, kRowShl4 = 0x104, kQuadXor2 = 0x4E, kQuadXor1 = 0xB1;
template <int CTRL>
__device__ __forceinline__ double dpp_partner(double v) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = dpp_word<CTRL>((unsigned)u), hi = dpp_word<CTRL>((unsigned)(u >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <int CTRL>
__device__ __forceinline__ float dpp_partner(float v) {
  return __uint_as_float(dpp_word<CTRL>(__float_as_uint(v)));
}
// v and w exchanged between the lanes of each pair: the lower lane ends with both
// lanes' v in a and b, the upper one with both lanes' w
template <int FAR>
__device__ __forceinline__ void swap_two(unsigned v, unsigned w, unsigned &a, unsigned &b) {
  if constexpr (FAR == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, w, false, false);
    a = r[0];
    b = r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane16_swap(v, w, false, false);
    a = r[0];
    b = r[1];
  }
}
template <int FAR>
__device__ __forceinline__ void lane_pair(double v, double &a, double &b) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  unsigned al, ah, bl, bh;
  swap_two<FAR>((unsigned)u, (unsigned)u, al, bl);
  swap_two<FAR>((unsigned)(u >> 32), (unsigned)(u >> 32), ah, bh);
  a = __longlong_as_double((long long)(((unsigned long long)ah << 32) | al));
  b = __longlong_as_double((long long)(((unsigned long long)bh << 32) | bl));
}
template <int FAR>
__device__ __forceinline__ void lane_pair(float v, float &a, float &b) {
  unsigned ua, ub;
  swap_two<FAR>(__float_as_uint(v), __float_as_uint(v), ua, ub);
  a = __uint_as_float(ua);
  b = __uint_as_float(ub);
}
// A step of a reduce-scatter: the lower lane of a pair returns both lanes' v, the upper
// one both lanes' w.
template <int FAR>
__device__ __forceinline__ float lane_swap_add(float v, float w) {
  unsigned a, b;
  swap_two<FAR>(__float_as_uint(v), __float_as_uint(w), a, b);
  return __uint_as_float(a) + __uint_as_float(b);
}
template <int FAR>
__device__ __forceinline__ double lane_swap_add(double v, double w) {
  const unsigned long long p = (unsigned long long)__double_as_longlong(v);
  const unsigned long long q = (unsigned long long)__double_as_longlong(w);
  unsigned al, ah, bl, bh;
  swap_two<FAR>((unsigned)p, (unsigned)q, al, bl);
  swap_two<FAR>((unsigned)(p >> 32), (unsigned)(q >> 32), ah, bh);
  return __longlong_as_double((long long)(((unsigned long long)ah << 32) | al)) +
         __longlong_as_double((long long)(((unsigned long long)bh << 32) | bl));
}
// op over the wave, in every lane (op commutative: the pairs are those of the butterfly
// with offsets 32, 16, 8, 4, 2, 1)
template <typename T, typename Op>
__device__ __forceinline__ T wave_reduce(T v, Op op) {
  T a, b;
  lane_pair<32>(v, a, b);
  v = op(a, b);
  lane_pair<16>(v, a, b);
  v = op(a, b);
  v = op(v, dpp_partner<kRowRor8>(v));
  v = op(v, dpp_partner<kRowRor4>(v));
  v = op(v, dpp_partner<kQuadXor2>(v));
  return op(v, dpp_partner<kQuadXor1>(v));
}
__device__ __forceinline__ double wave_sum(double v) {
  return wave_reduce(v, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ float wave_sum_f(float v) {
  return wave_reduce(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ double wave_min(double v) {
  return wave_reduce(v, [](double a, double b) { return fmin(a, b); });
}
__device__ __forceinline__ double wave_max(double v) {
  return wave_reduce(v, [](double a, double b) { return fmax(a, b); });
}

// Sum of one double over a block (each wave's butterfly sum, then the waves in
// order: a fixed order), written as a 4-wide partial (value, 0, 0, 0) at
// out[4 * blockIdx.x].  Called by every thread of the block.
__device__ __forceinline__ void block_sum4_dev(double v0, double *out) {
  __shared__ double s[16];  // one sum per wave (blocks of up to 1024 threads)
  const double w = wave_sum(v0);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = w;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) t += s[k];
    out[4 * blockIdx.x + 0] = t;
    out[4 * blockIdx.x + 1] = 0.0;
    out[4 * blockIdx.x + 2] = 0.0;
    out[4 * blockIdx.x + 3] = 0.0;
  }
}

// The largest displacement since the last prune is kept as kDmaxSpread words
// (float bits, max-combined) kDmaxStride words apart, two sets alternating by step.
constexpr int kDmaxSpread = 64;
constexpr int kDmaxStride = 16;

// The next MD step's opening work done by an integrator kernel for its atom,
// when that step keeps the list (k_begin_nb does it otherwise): the new
// position into the slot arrays, its displacement since the last prune folded
// into the next evaluation's set of maxima, the other set cleared, and the
// force accumulators cleared once the integrator has read them.
// Without the nonbonded term (spos null) only the accumulators are cleared.
struct OpenNext {
  int on;
  int cur;  // the set of maxima of the next evaluation
  SlotPos *spos;
  float4 *spos32;
  const SlotPos *pref;
  unsigned *dmax;
  long long *nbx, *nby, *nbz, *fbx, *fby, *fbz;
};

// Called by every thread of an integrator kernel (O.on is uniform); i is the
// thread's atom, s its slot, r its position at the last prune (O.pref[s],
// loaded by the caller with its other loads), (px, py, pz) its new position.
__device__ __forceinline__ void open_next_at(const OpenNext &O, int i, int n, int s, const SlotPos &r,
                                             double px, double py, double pz) {
  if (!O.spos) {
    if (i < n) {
      O.fbx[i] = 0;
      O.fby[i] = 0;
      O.fbz[i] = 0;
    }
    return;
  }
  double d = 0.0;
  if (i < n) {
    SlotPos p;
    p.x = px;
    p.y = py;
    p.z = pz;
    p.pad = 0.0;
    const double dx = px - r.x, dy = py - r.y, dz = pz - r.z;
    d = sqrt(dx * dx + dy * dy + dz * dz);
    if (!(d == d)) d = 3.0e38;  // NaN positions force a prune
    O.spos[s] = p;
    O.spos32[s] = make_float4((float)px, (float)py, (float)pz, 0.0f);
    O.nbx[s] = 0;
    O.nby[s] = 0;
    O.nbz[s] = 0;
    O.fbx[i] = 0;
    O.fby[i] = 0;
    O.fbz[i] = 0;
  }
  if (i < kDmaxSpread) O.dmax[((1 - O.cur) * kDmaxSpread + i) * kDmaxStride] = 0u;
  d = wave_max(d);
  if ((threadIdx.x & 63) == 0 && d > 0.0)
    atomicMax(&O.dmax[(O.cur * kDmaxSpread + (blockIdx.x % kDmaxSpread)) * kDmaxStride],
              __float_as_uint((float)(d * (1.0 + 1e-6))));
}

// The same, loading the slot and the prune position itself.
__device__ __forceinline__ void open_next(const OpenNext &O, int i, int n, const int *__restrict__ orig_slot,
                                          double px, double py, double pz) {
  int s = 0;
  SlotPos r{};
  if (i < n && O.spos) {
    s = orig_slot[i];
    r = O.pref[s];
  }
  open_next_at(O, i, n, s, r, px, py, pz);
}

// Sums of 4-wide energy partials, all lists at once, by one workgroup; each
// list is summed in a fixed order (thread-strided partial sums, then each wave,
// then the wave sums in wave order). Then, for an MD step, the step's trace
// entry: trace[2*s] = epot (J), trace[2*s+1] = ekin (J) from e_out (kcal/mol, 4 doubles
// per component slot; the kinetic energy slot is in J).
// Run by one whole workgroup of kSumThreads threads (every thread calls it).
// LEAN sums the lists one after another with few registers (for a workgroup of
// a kernel whose own work hides the latency); the additions are the same, in
// the same order, so both forms give the same bits.
template <bool LEAN = false>
__device__ __forceinline__ void sum_lists(const SumList &L) {
  constexpr int T = kSumThreads;
  constexpr int W = T / 64;
  __shared__ double s[W][kMaxSums][4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if constexpr (LEAN) {
    for (int e = 0; e < L.n; e++) {
      const double4 *P = reinterpret_cast<const double4 *>(L.part[e]);
      const int cnt = L.count[e];
      double a[4] = {0.0, 0.0, 0.0, 0.0};
      int i = threadIdx.x;
      if (i < cnt) {
        const double4 v = P[i];
        a[0] = v.x;
        a[1] = v.y;
        a[2] = v.z;
        a[3] = v.w;
      }
      for (i += T; i + 3 * T < cnt; i += 4 * T) {
        double4 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = P[i + u * T];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          a[0] += v[u].x;
          a[1] += v[u].y;
          a[2] += v[u].z;
          a[3] += v[u].w;
        }
      }
      for (; i < cnt; i += T) {
        const double4 v = P[i];
        a[0] += v.x;
        a[1] += v.y;
        a[2] += v.z;
        a[3] += v.w;
      }
#pragma unroll
      for (int d = 0; d < 4; d++) {
        const double t = wave_sum(a[d]);
        if (lane == 0) s[w][e][d] = t;
      }
    }
  } else {
  // each thread issues its first load of every list before any use, so the
  // lists' global loads are in flight together; longer lists continue in a loop
  double4 first[kMaxSums];
#pragma unroll
  for (int e = 0; e < kMaxSums; e++) {
    first[e] = make_double4(0.0, 0.0, 0.0, 0.0);
    if (e < L.n && (int)threadIdx.x < L.count[e])
      first[e] = reinterpret_cast<const double4 *>(L.part[e])[threadIdx.x];
  }
  double a[kMaxSums][4];
#pragma unroll
  for (int e = 0; e < kMaxSums; e++) {
    a[e][0] = first[e].x;
    a[e][1] = first[e].y;
    a[e][2] = first[e].z;
    a[e][3] = first[e].w;
    if (e < L.n) {
      const double4 *P = reinterpret_cast<const double4 *>(L.part[e]);
      int i = threadIdx.x + T;
      for (; i + 3 * T < L.count[e]; i += 4 * T) {  // four loads in flight, added in order
        double4 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = P[i + u * T];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          a[e][0] += v[u].x;
          a[e][1] += v[u].y;
          a[e][2] += v[u].z;
          a[e][3] += v[u].w;
        }
      }
      for (; i < L.count[e]; i += T) {
        const double4 v = P[i];
        a[e][0] += v.x;
        a[e][1] += v.y;
        a[e][2] += v.z;
        a[e][3] += v.w;
      }
    }
  }
#pragma unroll
  for (int e = 0; e < kMaxSums; e++) {
    if (e < L.n) {
      for (int d = 0; d < 4; d++) {
        const double t = wave_sum(a[e][d]);
        if (lane == 0) s[w][e][d] = t;
      }
    }
  }
  }
  __syncthreads();
  if (threadIdx.x < 4 * kMaxSums) {
    const int e = threadIdx.x >> 2, d = threadIdx.x & 3;
    if (e < L.n) {
      double t = 0.0;
      for (int k = 0; k < W; k++) t += s[k][e][d];
      L.out[e][d] = t;
    }
  }
  __syncthreads();
  if (L.record && threadIdx.x == 0) {
    const double *E = L.e_out;
    const StepRecord &R = L.rec;
    double ep = 0.0;
    if (R.use_sasa) ep += E[13];
    if (R.use_nb) ep += E[0] + E[1] + R.vdwcor;
    if (R.use_bonded) ep += E[4] + E[5] + E[6];
    if (R.use_gb) ep += E[8] + E[9] + E[10] + E[12];
    R.trace[2 * R.step] = ep * R.kcal_to_J;
    R.trace[2 * R.step + 1] = E[20];
  }
}

// GB's energy sums: `which` 0 sums system sysi's 4-wide tile-pair partials into slots
// off .. off + slots - 1, 1 its self energies into slot off + 4 (thread-strided sums, then a
// tree).  Run by a whole workgroup of 256 threads; s: 4 x 256 doubles of LDS.
__device__ __forceinline__ void gb_sums_block(const GBSums &G, int sysi, int which, double (*s)[256]) {
  double *out = G.out + (size_t)sysi * G.stride + G.off;
  if (which == 0) {
    double a[4] = {0, 0, 0, 0};
    for (int k = G.beg[sysi] + threadIdx.x; k < G.end[sysi]; k += 256)
      for (int d = 0; d < 4; d++) a[d] += G.part[4 * k + d];
    for (int d = 0; d < 4; d++) s[d][threadIdx.x] = a[d];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
      if ((int)threadIdx.x < w)
        for (int d = 0; d < 4; d++) s[d][threadIdx.x] += s[d][threadIdx.x + w];
      __syncthreads();
    }
    if ((int)threadIdx.x < G.slots) out[threadIdx.x] = s[threadIdx.x][0];
  } else {
    double a = 0.0;
    for (int k = threadIdx.x; k < G.count[sysi]; k += 256) a += G.eself[G.first[sysi] + k];
    s[0][threadIdx.x] = a;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
      if ((int)threadIdx.x < w) s[0][threadIdx.x] += s[0][threadIdx.x + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) out[4] = s[0][0];
  }
}

// Runs fn on the engine behind a C-ABI handle with its device current, turning
// exceptions into PD-style error codes (the message is kept for pdgpu_last_error).
template <typename F>
inline int guarded(pdgpu_engine *h, F &&fn) {
  Engine *e = reinterpret_cast<Engine *>(h);
  if (!e) return PDGPU_ERR_ARG;
  try {
    PDGPU_HIP(hipSetDevice(e->device));
    fn(*e);
    return PDGPU_OK;
  } catch (const EngineError &x) {
    e->last_error = x.what();
    return x.code;
  } catch (const std::bad_alloc &) {
    e->last_error = "host allocation failed";
    return PDGPU_ERR_NOMEM;
  } catch (const std::exception &x) {
    e->last_error = x.what();
    return PDGPU_ERR_ARG;
  }
}

}  // namespace pdgpu
