// k_nonbonded.hip -- FF_NonBonded::calcForces on the device.
//
// Restates FF_NonBonded_CalcForces_T_fast2 (nonbonded.cpp:559-910) over the
// cluster list built by k_list.hip.  A workgroup takes one work group of up to
// four consecutive i-clusters of a grid column, one wavefront per i-cluster
// (8 atoms, held in scalar registers).  The 64 lanes of a wave walk the
// cluster's list entries, one j atom per lane, and loop over the 8 i atoms.
// Per pair:
//   * the displacement from FP64 positions relative to the i-cluster's first
//     atom c: d = ((p_j - c) + basis[image]) - (p_i - c), rounded to FP32 once;
//   * PD's cutoff test r^2 <= Cutoff^2 (nonbonded.cpp:718-722): decided from the
//     FP32 r^2 whenever it lies more than kNearBand from Cutoff^2 (VdwCutoff^2),
//     far beyond the FP32 error, and otherwise recomputed in FP64 exactly as PD
//     does, d = (p_j - p_i) + basis[image], r^2 = (x*x + y*y) + z*z; so the
//     interacting pair set of every step is PD's, bit for bit;
//   * the pair energy/force in FP32 (kcal/mol, A) with PD's expressions:
//     LJ 2eps(A/2 - B) with its energy switch (always on, nonbonded.cpp:748-761),
//     Coulomb plain / energy-switched / force-switched (nonbonded.cpp:766-821);
//   * 1-2/1-3 pairs (scale 0) drop out, 1-4 pairs use Vdw14/Elec14Scaling
//     (nonbonded.cpp:650-651).
// Forces are 64-bit fixed point.  Atomics to global memory run at a bounded
// rate per lane operation on this GPU, so the j forces of the workgroup are
// first summed in LDS: every list entry carries the rank of its j-cluster in
// the work group's candidate table, and at the end the workgroup adds each
// touched slot of the table to global memory once.  Integer adds are
// order-independent, so the forces are bitwise reproducible.  Energies go to
// per-wave FP64 partials reduced in a fixed order.
//
// Small systems (size_eval_buffers draws the line) run the same rounds in FP64, two
// waves to a cluster: their launches wait for latency, not issue, so the wider
// arithmetic is nearly free and the split pays for it.  512 waters: 28.4 us a launch
// with one FP32 wave a cluster, 13 now, and the errors of 50 MD steps against 64 bits
// 100 to 1,000 times smaller.  A chip-filling launch (98,304 atoms, 95 us) is bound
// by issue; there the flush without a division per slot, the lane swaps and DPP sums
// of the epilogue and the energy sums in a workgroup of their own took it from 101.
#include "bonded_dev.hpp"
#include "engine.hpp"
#include "group_order_dev.hpp"

#include <type_traits>

#include <cmath>

namespace pdgpu {

namespace {

enum { EL_NONE = 0, EL_PLAIN = 1, EL_ESWITCH = 3, EL_FSWITCH = 4 };

// |r^2_fp32 - r^2_exact| is below 1e-5 r^2 (one FP32 rounding of d, three of the
// sum); pairs within this band of a cutoff are re-tested in FP64.
constexpr float kNearBand = 0.01f;
// The FP64 pair arithmetic's r^2 differs from PD's by a few ulp of the coordinates times
// r: 1e-12 A^2 in a 100 A box, 1e-6 at coordinates of 1e8 A.
constexpr double kFineBand = 1e-5;

// Image index (i+1)*9 + (j+1)*3 + (k+1) -> the basis vector (i*Lx, j*Ly, k*Lz)
// of PeriodicBox::setupCellDimensions (space.cpp:94-109).
__device__ __forceinline__ double image_shift(int img, int axis, double L) {
  int k = axis == 0 ? img / 9 : (axis == 1 ? (img / 3) % 3 : img % 3);
  return k == 1 ? 0.0 : (k == 2 ? L : -L);
}

// First kernel of an evaluation with the nonbonded term.  Gathers the FP64
// positions into slot order, folds each atom's displacement since the last
// prune into this evaluation's set of spread maxima (the other set is cleared
// for the next evaluation) and clears the force accumulators and energy slots.
__global__ void k_begin_nb(int nslots, int n, const int *__restrict__ n_clusters, const int *__restrict__ slot_orig,
                           const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
                           SlotPos *__restrict__ spos, float4 *__restrict__ spos32, const SlotPos *__restrict__ pref,
                           unsigned *__restrict__ dmax,
                           int cur, long long *__restrict__ nbx, long long *__restrict__ nby,
                           long long *__restrict__ nbz, long long *__restrict__ fbx, long long *__restrict__ fby,
                           long long *__restrict__ fbz, double *__restrict__ e_out, int n_e, int zero_e,
                           SumList L) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (dmax && s < kDmaxSpread) dmax[((1 - cur) * kDmaxSpread + s) * kDmaxStride] = 0u;
  if (zero_e && s < n_e) e_out[s] = 0.0;
  if (s < n) {
    fbx[s] = 0;
    fby[s] = 0;
    fbz[s] = 0;
  }
  double d = 0.0;
  if (s < nslots) {
    nbx[s] = 0;
    nby[s] = 0;
    nbz[s] = 0;
    if (s < *n_clusters * kClusterSize) {
      const int a = slot_orig[s];
      SlotPos p;
      if (a >= 0) {
        p.x = x[a];
        p.y = y[a];
        p.z = z[a];
        const SlotPos r = pref[s];
        const double dx = p.x - r.x, dy = p.y - r.y, dz = p.z - r.z;
        d = sqrt(dx * dx + dy * dy + dz * dz);
        if (!(d == d)) d = 3.0e38;  // NaN positions force a prune
      } else {  // padding slot: far away, zero parameters, never listed
        p.x = 1.0e6;
        p.y = 1.0e6;
        p.z = 1.0e6;
      }
      p.pad = 0.0;
      spos[s] = p;
      spos32[s] = make_float4((float)p.x, (float)p.y, (float)p.z, 0.0f);
    }
  }
  d = wave_max(d);
  // rounded up (float bits of non-negative values order like the values)
  // one atomic per wave, spread over kDmaxSpread words on separate cache lines:
  // device-scope atomics on one address serialise
  if ((threadIdx.x & 63) == 0 && d > 0.0)
    atomicMax(&dmax[(cur * kDmaxSpread + (blockIdx.x % kDmaxSpread)) * kDmaxStride],
              __float_as_uint((float)(d * (1.0 + 1e-6))));
  // the previous MD step's energy sums and trace entry (their partials are not
  // written again before this step's force kernels, which follow this one)
  if (blockIdx.x == 0 && (L.n > 0 || L.record)) sum_lists(L);
}

// Rolling prune of the list: keeps the pairs within Cutoff + margin at the
// current positions.  A pair left out is more than margin - 2 * dmax beyond the
// cutoff at any later step, so while 2 * dmax stays below margin (minus a
// rounding allowance) the pruned list holds every pair within the cutoff; the
// kernel returns at once in that case.  One wave per i-cluster, entries kept in
// their order.
// Four i-clusters per workgroup, one wave each; a wave takes 256 entries per
// round (four per lane) with every load of the round issued before the tests.
constexpr int kPruneDepth = 4;
constexpr int kPruneWaves = 4;  // i-clusters (one wave each) per workgroup
__global__ __launch_bounds__(64 * kPruneWaves) void k_prune(const int *__restrict__ n_clusters, double Lx, double Ly, double Lz,
                                               float rk2, float margin_ok, int forced,
                                               const unsigned *__restrict__ dmax,  // this evaluation's words
                                               const SlotPos *__restrict__ spos, const float4 *__restrict__ spos32,
                                               const uint2 *__restrict__ entries,
                                               const int *__restrict__ cl_count, int stride,
                                               uint2 *__restrict__ pentries, int *__restrict__ pcount,
                                               int *__restrict__ pcount_nolj, SlotPos *__restrict__ pref,
                                               GroupOrderArgs G) {
  // after a list build, the last workgroup computes the nonbonded kernel's
  // dispatch order (the forced prune of the other workgroups hides it)
  if (G.on && blockIdx.x == gridDim.x - 1) {
    group_order_block(G.max_groups, G.n_groups, G.per_cap, G.gwork, G.order);
    return;
  }
  __shared__ float shtab[27 * 3];
  __shared__ unsigned s_dmax;
  if (threadIdx.x < 64) {  // the largest of the spread words
    unsigned v = threadIdx.x < kDmaxSpread ? dmax[threadIdx.x * kDmaxStride] : 0u;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = max(v, (unsigned)__shfl_xor((int)v, off, 64));
    if (threadIdx.x == 0) s_dmax = v;
  }
  __syncthreads();
  if (!forced && 2.0f * __uint_as_float(s_dmax) <= margin_ok) return;
  for (int t = threadIdx.x; t < 81; t += blockDim.x) {  // 27 images x 3 axes, whatever the block size
    const int axis = t % 3;
    shtab[t] = (float)image_shift(t / 3, axis, axis == 0 ? Lx : (axis == 1 ? Ly : Lz));
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int ci = blockIdx.x * kPruneWaves + (threadIdx.x >> 6);
  if (ci >= *n_clusters) return;  // whole waves; no barrier follows
  if (lane < kClusterSize) pref[ci * kClusterSize + lane] = spos[ci * kClusterSize + lane];
  // FP32 positions and offsets from the cluster's first atom: their rounding
  // (~1e-5 A at 100 A) is far inside the 1e-3 A allowance of the prune criterion
  const float4 oi = spos32[ci * kClusterSize];
  float iox[8], ioy[8], ioz[8];
#pragma unroll
  for (int a = 0; a < 8; a++) {
    const float4 p = spos32[ci * kClusterSize + a];
    iox[a] = p.x - oi.x;
    ioy[a] = p.y - oi.y;
    ioz[a] = p.z - oi.z;
  }
  const int cnt = cl_count[ci];
  const uint2 *E = entries + (size_t)ci * stride;
  uint2 *PE = pentries + (size_t)ci * stride;
  // entries whose j atom has an LJ epsilon go to the front, the others to the
  // back (last one first), so the nonbonded kernel runs whole rounds without LJ
  int out = 0, out_nolj = 0;
  for (int k0 = 0; k0 < cnt; k0 += 64 * kPruneDepth) {
    uint2 ent[kPruneDepth];
    float4 pj[kPruneDepth];
#pragma unroll
    for (int u = 0; u < kPruneDepth; u++) {
      const int k = k0 + 64 * u + lane;
      ent[u] = k < cnt ? E[k] : make_uint2(0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < kPruneDepth; u++) {
      const int k = k0 + 64 * u + lane;
      if (k < cnt) pj[u] = spos32[ent[u].x & 0xFFFFFFu];
    }
#pragma unroll
    for (int u = 0; u < kPruneDepth; u++) {
      const int k = k0 + 64 * u + lane;
      unsigned keep = 0u;
      if (k < cnt) {
        const int img = (int)((ent[u].x >> 24) & 31u);
        const float ax = (pj[u].x - oi.x) + shtab[3 * img], ay = (pj[u].y - oi.y) + shtab[3 * img + 1],
                    az = (pj[u].z - oi.z) + shtab[3 * img + 2];
#pragma unroll
        for (int a = 0; a < 8; a++) {
          const float dx = ax - iox[a], dy = ay - ioy[a], dz = az - ioz[a];
          keep |= ((dx * dx + dy * dy + dz * dz) <= rk2 ? 1u : 0u) << a;
        }
        keep &= ent[u].y & 0xFFu;
      }
      const bool jlj = (ent[u].x >> 29) & 1u;
      const unsigned long long below = (1ull << lane) - 1ull;
      const unsigned long long b = __ballot(keep != 0u && jlj), bn = __ballot(keep != 0u && !jlj);
      const uint2 e = make_uint2(ent[u].x, (ent[u].y & ~0xFFu) | keep);
      if (keep && jlj) PE[out + __popcll(b & below)] = e;
      if (keep && !jlj) PE[stride - 1 - (out_nolj + __popcll(bn & below))] = e;
      out += __popcll(b);
      out_nolj += __popcll(bn);
    }
  }
  if (lane == 0) {
    pcount[ci] = out;
    pcount_nolj[ci] = out_nolj;
  }
}


__device__ __forceinline__ void lds_fix_add(long long *p, long long v) {
  atomicAdd(reinterpret_cast<unsigned long long *>(p), static_cast<unsigned long long>(v));
}

constexpr int kMaxShare = 2;  // nb_share at most

template <int ELEC, bool VDW, bool FORCES, bool FINE>
__global__ __launch_bounds__(64 * kGroup * kMaxShare) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_nonbonded(
    NBKernelParams P, int n_order, int max_groups, int parts, const int *__restrict__ n_groups, const int *__restrict__ grp_order,
    const int *__restrict__ grp_first,
    const int *__restrict__ grp_count, const int *__restrict__ wg_ncand, const int *__restrict__ wg_cand,
    double Lx, double Ly, double Lz, const SlotPos *__restrict__ spos, const float4 *__restrict__ sprm,
    const float4 *__restrict__ sprm_lo,
    const uint2 *__restrict__ entries,
    int stride, const int *__restrict__ cl_count, const int *__restrict__ cl_count_nolj,
    long long *__restrict__ fx, long long *__restrict__ fy,
    long long *__restrict__ fz, double *__restrict__ e_partial, SumList L, BondedArrays B, int n_bonded_blocks,
    const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
    long long *__restrict__ fbx, long long *__restrict__ fby, long long *__restrict__ fbz,
    double *__restrict__ e_partial_bonded) {
  // the previous MD step's energy sums and trace entry, in a workgroup of their own:
  // the partials they read are not written by this kernel (its own go to the
  // other of two alternating arrays), and the rest of the grid hides their latency
  const bool sums = L.n > 0 || L.record;
  if (sums && blockIdx.x == gridDim.x - 1) {
    if (threadIdx.x < kSumThreads) sum_lists<true>(L);  // whole waves leave: its barriers wait for the others only
    return;
  }
  __shared__ __align__(16) long long jacc[3][kGroupRanks * kClusterSize];
  __shared__ int cand[kGroupRanks];
  __shared__ double shtab[27 * 3];
  // i atoms: offset from the cluster's first atom, in FP32 or (FINE) FP64
  using Off = std::conditional_t<FINE, SlotPos, float4>;
  __shared__ Off ioff[kGroup][kClusterSize];
  __shared__ Off iprm[kGroup][kClusterSize];     // i atoms: q, LJ radius, sqrt(eps)
  __shared__ double s_e[kGroup * kMaxShare][3];
  // The last n_bonded_blocks workgroups take FF_Bonded's terms of the same
  // evaluation (dispatched last, they fill the CUs the ending nonbonded
  // workgroups leave idle), with the j-force table's LDS as their window.
  const int nblk = (int)gridDim.x - n_bonded_blocks - (sums ? 1 : 0);
  if ((int)blockIdx.x >= nblk) {
    if (threadIdx.x >= kBondedThreads) return;  // whole waves
    bonded_block((int)blockIdx.x - nblk, B, x, y, z, fbx, fby, fbz, e_partial_bonded, nullptr, &jacc[0][0]);
    return;
  }
  // the group of this workgroup: each XCD takes a contiguous run of (spatially
  // adjacent) groups of equal total work, heaviest first (the order the list
  // build computed)
  const int part = (int)blockIdx.x / n_order;
  const int g = grp_order[(int)blockIdx.x - part * n_order];
  if (g < 0) return;  // a block no group uses
  e_partial += 4 * (g + part * max_groups);
  // `wave` is the cluster's place in the group; part: this workgroup takes rounds part,
  // part + parts, ... of each of its clusters
  const int wave_id = threadIdx.x >> 6, wave = wave_id & (kGroup - 1);
  const int lane = threadIdx.x & 63;
  if (g >= *n_groups) {  // padding: the whole workgroup leaves together
    if (threadIdx.x < 4) e_partial[threadIdx.x] = 0.0;
    return;
  }
  const int nr = wg_ncand[g];
  for (int t = threadIdx.x; t < 3 * kGroupRanks * kClusterSize / 2; t += blockDim.x)
    reinterpret_cast<longlong2 *>(&jacc[0][0])[t] = make_longlong2(0, 0);
  for (int t = threadIdx.x; t < nr; t += blockDim.x) cand[t] = wg_cand[(size_t)g * kGroupStride + t];
  if (threadIdx.x < 81) {
    const int axis = threadIdx.x % 3;
    shtab[threadIdx.x] = image_shift(threadIdx.x / 3, axis, axis == 0 ? Lx : (axis == 1 ? Ly : Lz));
  }
  const int nc = grp_count[g], c0 = grp_first[g];
  if ((int)threadIdx.x >= 128 && (int)threadIdx.x < 128 + nc * kClusterSize) {  // the third wave (shtab: the first two)
    const int a = threadIdx.x - 128, s = c0 * kClusterSize + a;
    const SlotPos p = spos[s], o = spos[s & ~(kClusterSize - 1)];
    if constexpr (FINE)
      (&ioff[0][0])[a] = SlotPos{p.x - o.x, p.y - o.y, p.z - o.z, 0.0};
    else
      (&ioff[0][0])[a] = make_float4((float)(p.x - o.x), (float)(p.y - o.y), (float)(p.z - o.z), 0.0f);
    const float4 q = sprm[s];
    if constexpr (FINE) {
      const float4 l = sprm_lo[s];
      (&iprm[0][0])[a] = SlotPos{(double)q.x + l.x, (double)q.y + l.y, (double)q.z + l.z, 0.0};
    } else {
      (&iprm[0][0])[a] = q;
    }
  }
  __syncthreads();

  double ev = 0.0, ee = 0.0, vir = 0.0;  // per-lane FP64 energy accumulators
  if (wave < nc) {
    // uniform over the wave: the i-cluster data below lives in scalar registers
    const int ci = __builtin_amdgcn_readfirstlane(c0 + wave);
    const SlotPos oi = spos[ci * kClusterSize];  // the cluster's first atom (always a real atom)
    // The column sort puts a cluster's atoms with an LJ epsilon first; a cluster
    // whose slots 4..7 hold none (water: its hydrogens) skips LJ for them.
    // slots 0..lj_need-1 hold every atom of the cluster with an LJ epsilon
    const unsigned lj_mask = (unsigned)__ballot(iprm[wave][lane & (kClusterSize - 1)].z != 0) & 0xFFu;
    const int lj_need = 32 - __clz((int)lj_mask);
    // FINE: two waves share the cluster, each with every other of its atoms
    constexpr int kOwn = FINE ? 4 : 8;
    const int half = FINE ? __builtin_amdgcn_readfirstlane(wave_id / kGroup) : 0;
    std::conditional_t<FINE, double, float> fix[kOwn], fiy[kOwn], fiz[kOwn];
#pragma unroll
    for (int a = 0; a < kOwn; a++) fix[a] = fiy[a] = fiz[a] = 0;
    const float cut2f = (float)P.cut2, vcut2f = (float)P.vdwcut2;

    // the pruned entries: those whose j atom has an LJ epsilon from the front of
    // the cluster's run, then the others from its back (last one first); rounds
    // past the first group run without LJ arithmetic
    const int cnt_lj = cl_count[ci];
    const int cnt = cnt_lj + cl_count_nolj[ci];
    const uint2 *E = entries + (size_t)ci * stride;
    auto at = [&](int k) { return k < cnt_lj ? k : stride - 1 - (k - cnt_lj); };
    int k0 = 64 * part;
    const int step = 64 * parts;
    uint2 nxt = k0 + lane < cnt ? E[at(k0 + lane)] : make_uint2(0u, 0u);
    using L0 = std::integral_constant<int, 0>;
    using L2 = std::integral_constant<int, 2>;
    using L3 = std::integral_constant<int, 3>;
    using L4 = std::integral_constant<int, 4>;
    using L8 = std::integral_constant<int, 8>;
    using Real = std::conditional_t<FINE, double, float>;
    auto add_j = [&](uint2 ent, long long vx, long long vy, long long vz) {
      const int j = (int)(ent.x & 0xFFFFFFu);
      const unsigned rank = ent.y >> 24;
      if (rank < (unsigned)kGroupRanks) {
        const int l = (int)rank * kClusterSize + (j & (kClusterSize - 1));
        lds_fix_add(&jacc[0][l], vx);
        lds_fix_add(&jacc[1][l], vy);
        lds_fix_add(&jacc[2][l], vz);
      } else {
        fix_add(&fx[j], vx);
        fix_add(&fy[j], vy);
        fix_add(&fz[j], vz);
      }
    };
    // A round in FP64: the expressions of the FP32 pair loop below, term by term, from
    // 1/r by one Newton step on the FP32 reciprocal root (to ~1e-14).
    auto fine_round = [&](auto lj_slots, uint2 ent, unsigned lm, float4 qj, double ax, double ay, double az) {
      if constexpr (FINE) {
        constexpr int NLJ = decltype(lj_slots)::value;
        const NBFine &D = P.d;
        lm = (lm >> half) & 0x55u;
        const unsigned codes = ((ent.y >> 8) & 0xFFFFu) >> (2 * half);
        const unsigned clo = codes & 0x5555u, chi = (codes >> 1) & 0x5555u;
        const unsigned excl = clo ^ chi, is14 = clo & chi;
        const float4 lo = sprm_lo[ent.x & 0xFFFFFFu];
        const double qjd = (double)qj.x + lo.x, rjd = (double)qj.y + lo.y, ejd = (double)qj.z + lo.z;
        double fjx = 0.0, fjy = 0.0, fjz = 0.0;
        int ib = wave * kClusterSize + half;
        asm volatile("" : "+v"(ib));
#pragma unroll
        for (int h = 0; h < 4; h++) {
          const int a = 2 * h;  // of this wave's half
          const SlotPos io = (&ioff[0][0])[ib + a], pa = (&iprm[0][0])[ib + a];
          const double dx = ax - io.x, dy = ay - io.y, dz = az - io.z;
          const double r2s = fma(dx, dx, fma(dy, dy, dz * dz));
          bool inc = r2s <= P.cut2, inv = r2s < P.vdwcut2;
          const bool listed = ((lm >> a) & 1u) && !((excl >> (2 * a)) & 1u);
          // PD's own test where the cutoff is near
          const bool near = fabs(r2s - P.cut2) < kFineBand || fabs(r2s - P.vdwcut2) < kFineBand;
          if (__builtin_expect(__ballot(near && listed) != 0ull, 0)) {
#pragma clang fp contract(off)
            const int j = (int)(ent.x & 0xFFFFFFu), img = (int)((ent.x >> 24) & 31u);
            const SlotPos pj = spos[j], pi = spos[ci * kClusterSize + half + a];
            const double ex = (pj.x - pi.x) + shtab[3 * img], ey = (pj.y - pi.y) + shtab[3 * img + 1],
                         ez = (pj.z - pi.z) + shtab[3 * img + 2];
            const double r2 = ex * ex + ey * ey + ez * ez;
            inc = r2 <= P.cut2;               // sqrdistij > sqrcutoff (nonbonded.cpp:722)
            inv = sqrt(r2) < P.vdwcut_d;      // Dist_ij < VdwCutoff (nonbonded.cpp:742)
          }
          const bool on = listed && inc;
          const bool s14 = (is14 >> (2 * a)) & 1u;
          const double r2 = on ? r2s : 1.0;
          double rinv = (double)__builtin_amdgcn_rsqf((float)r2);
          rinv = fma(0.5 * rinv, fma(-(r2 * rinv), rinv, 1.0), rinv);
          const double rinv2 = rinv * rinv;
          double dEdr = 0.0;
          if (VDW && h < NLJ) {
            const double eps_ij = (s14 ? D.vdw14 : 1.0) * (pa.z * ejd);
            const double eps = (on && inv) ? eps_ij : 0.0;
            const double Rij = pa.y + rjd;
            const double s2 = Rij * Rij * rinv2;
            const double B = s2 * s2 * s2;
            const double eB = eps * B;
            const double e0 = eB * (B - 2.0);
            const double d0 = (-12.0 * rinv) * fma(eB, B, -eB);
            const double t = fmax(fma(r2, rinv, -D.vdwinner), 0.0);
            const double u = D.invw_vdw * t;
            const double S0 = fma(-u, u, 1.0);
            const double S = S0 * S0;
            dEdr = fma(S, d0, e0 * (-D.invw2_vdw4 * t * S0));
            ev = fma(e0, S, ev);
          }
          if (ELEC != EL_NONE) {
            const double qq_ij = (s14 ? D.elec14 : 1.0) * (pa.x * qjd);
            const double qq = on ? qq_ij : 0.0;
            if (ELEC == EL_PLAIN) {
              const double e0 = qq * rinv;
              ee += e0;
              dEdr = fma(-e0, rinv, dEdr);
            } else if (ELEC == EL_ESWITCH) {
              const double e0 = qq * rinv;
              const double t = fmax(fma(r2, rinv, -D.inner), 0.0);
              const double u = D.invw_el * t;
              const double S0 = fma(-u, u, 1.0);
              const double S = S0 * S0;
              dEdr += fma(S, -e0 * rinv, e0 * (-D.invw2_el4 * t * S0));
              ee = fma(e0, S, ee);
            } else {
              const double x = fmin(fmax(fma(r2, D.fs_invw, D.fs_x0), 0.0), 1.0);
              const double S = fma(x * x, fma(2.0, x, -3.0), 1.0);
              const double poly = fma(r2, fma(r2, fma(D.fs_c4, r2, D.fs_c3), D.fs_c2), D.fs_c1);
              const double e_out = fma(-rinv, poly, D.fcut);
              const double e_in = rinv - D.eshift;
              ee = fma(qq, x > 0.0 ? e_out : e_in, ee);
              dEdr = fma(qq, -rinv2 * S, dEdr);
            }
          }
          const double sc = dEdr * rinv;
          if (FORCES) {
            fix[h] = fma(dx, sc, fix[h]);
            fiy[h] = fma(dy, sc, fiy[h]);
            fiz[h] = fma(dz, sc, fiz[h]);
            fjx = fma(-dx, sc, fjx);
            fjy = fma(-dy, sc, fjy);
            fjz = fma(-dz, sc, fjz);
          }
          vir = fma(r2, sc, vir);
        }
        if (FORCES && lm) add_j(ent, fix_from_double(fjx), fix_from_double(fjy), fix_from_double(fjz));
      }
    };
    // The rounds from k0 to k_end, with LJ arithmetic for slots 0..NLJ-1.  Each
    // LJ width has a round loop of its own (chosen once per cluster), so a
    // loop's only branch per round is whether its entries carry bond-order codes,
    // and the register allocator keeps the i-force partials in place through it
    // (one loop with every version behind a per-round switch copied them).
    auto rounds = [&](auto lj_slots, const int k_end) {
    for (; k0 < k_end; k0 += step) {
      const bool valid = k0 + lane < cnt;
      const uint2 ent = nxt;
      const int kn = k0 + step + lane;
      nxt = kn < cnt ? E[at(kn)] : make_uint2(0u, 0u);  // prefetch the next round
      const int j = (int)(ent.x & 0xFFFFFFu);
      const int img = (int)((ent.x >> 24) & 31u);
      const unsigned lm = valid ? (ent.y & 0xFFu) : 0u;
      const unsigned codes = (ent.y >> 8) & 0xFFFFu;
      const unsigned clo = codes & 0x5555u, chi = (codes >> 1) & 0x5555u;
      const unsigned excl = clo ^ chi;  // codes 1 and 2: 1-2 / 1-3 pairs, scale 0
      const unsigned is14 = clo & chi;  // code 3: 1-4 pair
      const float4 qj = sprm[j];
      // the j atom's image relative to the cluster's first atom: FP64, then FP32;
      // the pair displacements below are FP32 differences of FP32 offsets, within
      // ~1e-6 A of the FP64 displacement (the cutoff band below is 0.01 A^2 wide)
      Real ax, ay, az;
      {
        const SlotPos pj = spos[j];
        ax = (Real)((pj.x - oi.x) + shtab[3 * img]);
        ay = (Real)((pj.y - oi.y) + shtab[3 * img + 1]);
        az = (Real)((pj.z - oi.z) + shtab[3 * img + 2]);
      }
      if constexpr (FINE) {
        fine_round(lj_slots, ent, lm, qj, ax, ay, az);
        continue;
      } else {
      // -0.0f is the additive identity, so the first term of each sum needs no add
      float fjx = -0.0f, fjy = -0.0f, fjz = -0.0f;
      float ev8 = -0.0f, ee8 = -0.0f, vir8 = -0.0f;  // the 8 pairs of this entry
      // Re-read the i atoms from LDS in every round instead of holding 8 atoms in
      // registers: the empty asm hides that the index is loop-invariant.
      int ib = wave * kClusterSize;
      asm volatile("" : "+v"(ib));
      // cutoff decisions for the 8 pairs first, in FP32; a pair within kNearBand
      // of a cutoff takes PD's FP64 test (nonbonded.cpp:718-722) behind one
      // wave-uniform branch, rarely taken (also for pairs the entry does not list:
      // their decision is masked off later).  The displacements stay in registers
      // for the pair loop (each round loop has the registers to spare).
      float r2a[8], dxa[8], dya[8], dza[8];
      bool inca[8], inva[8];
      // the smallest distance of the 8 r^2 to a cutoff: one min per pair
      // instead of a flag per pair
      float mind = 2.0f * kNearBand;
      if (P.same_cut) {
        // one cutoff: outside the band r2 differs from it, so both tests agree
#pragma unroll
        for (int a = 0; a < 8; a++) {
          const float4 io = (&ioff[0][0])[ib + a];
          const float dx = ax - io.x, dy = ay - io.y, dz = az - io.z;
          dxa[a] = dx; dya[a] = dy; dza[a] = dz;
          r2a[a] = dx * dx + dy * dy + dz * dz;
          const float d = r2a[a] - cut2f;
          inca[a] = d <= 0.0f;
          inva[a] = inca[a];
          mind = fminf(mind, fabsf(d));
        }
      } else {
#pragma unroll
        for (int a = 0; a < 8; a++) {
          const float4 io = (&ioff[0][0])[ib + a];
          const float dx = ax - io.x, dy = ay - io.y, dz = az - io.z;
          dxa[a] = dx; dya[a] = dy; dza[a] = dz;
          r2a[a] = dx * dx + dy * dy + dz * dz;
          inca[a] = r2a[a] <= cut2f;
          inva[a] = r2a[a] < vcut2f;
          mind = fminf(mind, fminf(fabsf(r2a[a] - cut2f), fabsf(r2a[a] - vcut2f)));
        }
      }
      const bool anynear = mind < kNearBand;
      if (__builtin_expect(__ballot(anynear && lm != 0u) != 0ull, 0)) {
        const SlotPos pj = spos[j];
        const double shx = shtab[3 * img], shy = shtab[3 * img + 1], shz = shtab[3 * img + 2];
#pragma unroll
        for (int a = 0; a < 8; a++) {
          const bool near = fabsf(r2a[a] - cut2f) < kNearBand || fabsf(r2a[a] - vcut2f) < kNearBand;
          if (near && ((lm >> a) & 1u)) {
#pragma clang fp contract(off)
            const SlotPos pi = spos[ci * kClusterSize + a];
            const double ex = (pj.x - pi.x) + shx, ey = (pj.y - pi.y) + shy, ez = (pj.z - pi.z) + shz;
            const double r2 = ex * ex + ey * ey + ez * ez;
            inca[a] = r2 <= P.cut2;              // sqrdistij > sqrcutoff (nonbonded.cpp:722)
            inva[a] = sqrt(r2) < P.vdwcut_d;     // Dist_ij < VdwCutoff (nonbonded.cpp:742)
          }
        }
      }
      // The pair loop in six versions, chosen per round by wave-uniform tests:
      // rounds whose entries carry no bond-order code (no 1-2, 1-3 or 1-4 pair;
      // most rounds) skip decoding the codes, and the LJ arithmetic runs for
      // slots 0..NLJ-1 only: none when no j atom of the round (or no i atom)
      // has an epsilon, else 2, 3, 4 or 8 to cover the cluster's last slot that
      // holds one (the column sort puts them first).  A skipped LJ term would be
      // an exact zero, so every version gives the same bits.
      auto pair_loop = [&](auto has_codes, auto lj_slots) {
        constexpr bool HC = decltype(has_codes)::value;
        constexpr int NLJ = decltype(lj_slots)::value;  // LJ arithmetic for slots 0..NLJ-1
  #pragma unroll
        for (int a = 0; a < 8; a++) {
          const float dx = dxa[a], dy = dya[a], dz = dza[a], r2s_a = r2a[a];
          const bool inc = inca[a], inv = inva[a];
          const float4 pa = (&iprm[0][0])[ib + a];
          const bool on = ((lm >> a) & 1u) && (!HC || !((excl >> (2 * a)) & 1u)) && inc;
          const bool s14 = HC && ((is14 >> (2 * a)) & 1u);
          const float r2f = on ? r2s_a : 1.0f;
          const float rinv = __builtin_amdgcn_rsqf(r2f);
          const float r = r2f * rinv;
          const float rinv2 = rinv * rinv;
          // A pair that is off has eps = qq = 0, so every energy and force term below
          // comes out as (signed) zero without a select of its own.
          float dEdr = 0.0f, Ev = 0.0f, Ee = 0.0f;
          if (VDW && a < NLJ) {
            const float eps_ij = (s14 ? P.vdw14 : 1.0f) * pa.z * qj.z;
            // computed for every pair, then selected: a select of a product that
            // reads pa would be turned into a branch around the LDS read
            const float eps = (on && inv) ? eps_ij : 0.0f;
            const float Rij = pa.y + qj.y;
            const float s2 = Rij * Rij * rinv2;
            const float B = s2 * s2 * s2;  // A = B^2
            const float eB = eps * B;
            float e0 = eB * (B - 2.0f);                       // eps (A - 2B)
            float d0 = (-12.0f * rinv) * fmaf(eB, B, -eB);   // -12 eps (A - B) / r
            const float t = fmaxf(r - P.vdwinner, 0.0f);
            const float S0 = 1.0f - (P.invw_vdw * t) * (P.invw_vdw * t);
            const float dS = -P.invw2_vdw4 * t * S0;
            const float S = S0 * S0;
            d0 = S * d0 + e0 * dS;
            Ev = e0 * S;
            dEdr += d0;
          }
          if (ELEC != EL_NONE) {
            const float qq_ij = (s14 ? P.elec14 : 1.0f) * pa.x * qj.x;
            const float qq = on ? qq_ij : 0.0f;
            if (ELEC == EL_PLAIN) {
              Ee = qq * rinv;
              dEdr += -Ee * rinv;
            } else if (ELEC == EL_ESWITCH) {
              float e0 = qq * rinv;
              float d0 = -e0 * rinv;
              const float t = fmaxf(r - P.inner, 0.0f);
              const float S0 = 1.0f - (P.invw_el * t) * (P.invw_el * t);
              const float dS = -P.invw2_el4 * t * S0;
              const float S = S0 * S0;
              d0 = S * d0 + e0 * dS;
              Ee = e0 * S;
              dEdr += d0;
            } else {  // force switch (Steinbach & Brooks), nonbonded.cpp:798-819
              // outer: E = -qq (sA r (sB/r^2 + sC + sD r^2 + sE r^4) - fcut)
              //          = qq (fcut - c1/r - r (c2 + r^2 (c3 + c4 r^2))),
              //        dE/dr = -qq sA (rc^2 - r^2)^2 (rc^2 - 3 rin^2 + 2 r^2) / r^2
              // inner: E = qq (1/r - eshift), dE/dr = -qq / r^2
              // Both forces in one expression: with w = rc^2 - rin^2 and
              // x = (r^2 - rin^2) / w clamped to [0, 1], sA = 1/w^3 gives
              // sA (rc^2 - r^2)^2 (rc^2 - 3 rin^2 + 2 r^2) = (1-x)^2 (1+2x) = 1 - 3x^2 + 2x^3,
              // which is 1 inside rin.
              const float x = __builtin_amdgcn_fmed3f(fmaf(r2f, P.fs_invw, P.fs_x0), 0.0f, 1.0f);
              const float S = fmaf(x * x, fmaf(2.0f, x, -3.0f), 1.0f);
              const bool outer = x > 0.0f;  // r^2 > rin^2
              // c1/r + r (c2 + ...) = (c1 + r^2 (c2 + ...)) / r
              const float poly = fmaf(r2f, fmaf(r2f, fmaf(P.fs_c4, r2f, P.fs_c3), P.fs_c2), P.fs_c1);
              const float e_out = fmaf(-rinv, poly, P.fcut);
              const float e_in = rinv - P.eshift;
              Ee = qq * (outer ? e_out : e_in);
              dEdr = fmaf(qq, -rinv2 * S, dEdr);
            }
          }
          const float sc = dEdr * rinv;
          if (FORCES) {
            fix[a] = fmaf(dx, sc, fix[a]);
            fiy[a] = fmaf(dy, sc, fiy[a]);
            fiz[a] = fmaf(dz, sc, fiz[a]);
            fjx = fmaf(-dx, sc, fjx);
            fjy = fmaf(-dy, sc, fjy);
            fjz = fmaf(-dz, sc, fjz);
          }
          ev8 += Ev;
          ee8 += Ee;
          if (!FORCES) vir8 = fmaf(r2f, sc, vir8);  // r dE/dr (with forces: per entry, below)
        }
      };
      const bool anycodes = __ballot(codes != 0u) != 0ull;
      if (anycodes)
        pair_loop(std::true_type{}, lj_slots);
      else
        pair_loop(std::false_type{}, lj_slots);
      ev += (double)ev8;
      ee += (double)ee8;
      // The virial sum_a r_a dE/dr_a = sum_a d_a . g_a with g_a = d_a dE/dr / r (what
      // the i force of atom a gains) and d_a = A - o_a (A the j atom's offset, o_a
      // the i atom's): the entry adds A . sum_a g_a = -A . f_j, and the i atoms'
      // part sum o_a . g_a is taken once per cluster from the i-force partials.
      if (FORCES) vir8 = -fmaf(ax, fjx, fmaf(ay, fjy, az * fjz));
      vir += (double)vir8;
      if (FORCES && lm) add_j(ent, fix_from_float(fjx), fix_from_float(fjy), fix_from_float(fjz));
      }
    }
    };
    // rounds starting inside the entries with an LJ j atom take LJ for the
    // cluster's slots that hold an epsilon (none when no i atom has one); the
    // rest run without LJ arithmetic
    if constexpr (FINE) {
      const int need = (lj_need + 1 - half) / 2;  // of the half's four
      if (need == 0)
        rounds(L0{}, cnt_lj);
      else if (need <= 2)
        rounds(L2{}, cnt_lj);
      else
        rounds(L4{}, cnt_lj);
    } else {
      if (lj_need == 0)
        rounds(L0{}, cnt_lj);
      else if (lj_need <= 2)
        rounds(L2{}, cnt_lj);
      else if (lj_need == 3)
        rounds(L3{}, cnt_lj);
      else if (lj_need == 4)
        rounds(L4{}, cnt_lj);
      else
        rounds(L8{}, cnt_lj);
    }
    rounds(L0{}, cnt);
    // i forces: the cluster is rank `wave` of its own group's table.  The 24
    // per-lane partials (component-major: q = 8 * component + atom) are summed
    // over the wave by a reduce-scatter: each exchange step halves the values a
    // lane holds and the partner lane's half is added, so lane groups of 8 end
    // with 3 sums each, finished over the group (a fixed order throughout).
    if (FORCES) {
      if constexpr (!FINE) {
        // the i atoms' part of the virial: sum over the lane's entries of o_a . g_a
        double vi = 0.0;
#pragma unroll
        for (int a = 0; a < 8; a++) {
          const float4 io = ioff[wave][a];
          vi += (double)fmaf(io.x, fix[a], fmaf(io.y, fiy[a], io.z * fiz[a]));
        }
        vir -= vi;
      }
      // FINE: 12 values (q = 4 * component + atom), groups of 16 lanes ending with 3
      constexpr int V = 3 * kOwn;
      Real v[V], w[V / 2], u[V / 4];
#pragma unroll
      for (int a = 0; a < kOwn; a++) {
        v[a] = fix[a];
        v[kOwn + a] = fiy[a];
        v[2 * kOwn + a] = fiz[a];
      }
      const bool b5 = (lane & 32) != 0, b4 = (lane & 16) != 0, b3 = (lane & 8) != 0;
      // a swap leaves in a lane its own and its partner's term of the value it keeps
#pragma unroll
      for (int k = 0; k < V / 2; k++) w[k] = lane_swap_add<32>(v[k], v[V / 2 + k]);
#pragma unroll
      for (int k = 0; k < V / 4; k++) u[k] = lane_swap_add<16>(w[k], w[V / 4 + k]);
      Real s3[3];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        if constexpr (FINE)
          s3[k] = u[k] + dpp_partner<kRowRor8>(u[k]);
        else
          s3[k] = (b3 ? u[3 + k] : u[k]) + dpp_partner<kRowRor8>(b3 ? u[k] : u[3 + k]);
        s3[k] += dpp_partner<kRowShl4>(s3[k]);  // right in lanes 0..3 of each group of 8
        s3[k] += dpp_partner<kQuadXor2>(s3[k]);
        s3[k] += dpp_partner<kQuadXor1>(s3[k]);
      }
      if ((lane & (FINE ? 15 : 7)) == 0) {
        const int q0 = (b5 ? V / 2 : 0) + (b4 ? V / 4 : 0) + (!FINE && b3 ? 3 : 0);
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const int q = q0 + k;
          if constexpr (FINE)
            lds_fix_add(&jacc[q >> 2][wave * kClusterSize + 2 * (q & 3) + half], fix_from_double(s3[k]));
          else
            lds_fix_add(&jacc[q >> 3][wave * kClusterSize + (q & 7)], fix_from_float(s3[k]));
        }
      }
    }
  }
  // one energy partial per workgroup: the waves' sums in wave order
  const double sev = wave_sum(ev);
  const double see = wave_sum(ee);
  const double svir = wave_sum(vir);
  if (lane == 0) {
    s_e[wave_id][0] = sev;
    s_e[wave_id][1] = see;
    s_e[wave_id][2] = svir;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double t = 0.0;
    if (threadIdx.x < 3)
      for (int w = 0; w < (int)blockDim.x / 64; w++) t += s_e[w][threadIdx.x];
    e_partial[threadIdx.x] = t;
  }
  // flush the touched slots of the candidate table, consecutive threads on
  // consecutive slots of a j-cluster
  if (FORCES) {
    for (int l = threadIdx.x; l < nr * kClusterSize; l += blockDim.x) {
      const long long vx = jacc[0][l], vy = jacc[1][l], vz = jacc[2][l];
      if ((vx | vy | vz) == 0) continue;
      const int s = cand[l / kClusterSize] * kClusterSize + (l & (kClusterSize - 1));
      fix_add(&fx[s], vx);
      fix_add(&fy[s], vy);
      fix_add(&fz[s], vz);
    }
  }
}

// With bonded_partial the launch also runs the bonded terms in its last workgroups.
template <int ELEC, bool VDW, bool FORCES, bool FINE>
void launch(Engine &E, double *partial, const SumList &L, double *bonded_partial) {
  const int nbb = bonded_partial ? bonded_blocks(E.nbonds, E.nangles, E.ntors) : 0;
  const BondedArrays B = E.bonded_arrays();
  hipLaunchKernelGGL((k_nonbonded<ELEC, VDW, FORCES, FINE>), dim3(8 * E.nb_per_cap * E.nb_parts + nbb + (L.n > 0 || L.record ? 1 : 0)),
                     dim3(64 * kGroup * E.nb_share), 0, E.stream, E.nbk, 8 * E.nb_per_cap, E.max_groups, E.nb_parts, E.n_groups_d.p, E.grp_order.p, E.grp_first.p, E.grp_count.p, E.wg_ncand.p,
                     E.wg_cand.p,
                     E.periodic ? E.box[0] : 0.0, E.periodic ? E.box[1] : 0.0, E.periodic ? E.box[2] : 0.0,
                     E.spos.p, E.sprm.p, E.sprm_lo.p, E.pentries.p, (int)E.entry_capacity,
                     E.pcount.p, E.pcount_nolj.p, E.nbx.p, E.nby.p, E.nbz.p, partial, L, B, nbb, E.x.p, E.y.p,
                     E.z.p, E.fbx.p, E.fby.p, E.fbz.p, bonded_partial);
}

template <int ELEC>
void launch_mode(Engine &E, bool vdw, bool forces, double *partial, const SumList &L, double *bp) {
  // without forces: FF_NonBonded::calcEnergies_Full, the same kernel (nonbonded.cpp:1184-1202)
  auto go = [&](auto fine) {
    constexpr bool F = decltype(fine)::value;
    if (forces)
      vdw ? launch<ELEC, true, true, F>(E, partial, L, bp) : launch<ELEC, false, true, F>(E, partial, L, bp);
    else
      vdw ? launch<ELEC, true, false, F>(E, partial, L, bp) : launch<ELEC, false, false, F>(E, partial, L, bp);
  };
  E.nbk.fine ? go(std::true_type{}) : go(std::false_type{});
}

}  // namespace

void Engine::setup_nonbonded(const pdgpu_nb_params &p) {
  require(!h_charge.empty(), "atom parameters not set");
  // FF_NonBonded::setupBasisVectors refuses more than 32 image vectors (nonbonded.cpp:1059-1069);
  // PeriodicBox::setupCellDimensions(Cutoff) gives (2n+1)^3 vectors, n = ceil(Cutoff/half box).
  const double c = std::max(p.Cutoff, p.VdwCutoff);
  if (periodic) {
    for (int d = 0; d < 3; d++) {
      double nx = std::ceil(std::max(list_cutoff, c) / (box[d] / 2.0));
      if (nx > 1.0)
        throw EngineError(PDGPU_ERR_SETUP,
                          "FF_NonBonded: Cannot use more than 32 periodic boundary image vectors "
                          "(cutoff greater than half the periodic box width)");
    }
  }
  nb = p;
  list_cutoff = std::max(list_cutoff, c);  // NeighbourListBase::requestCutoff: the maximum wins
  NBKernelParams k{};
  const double C = p.Cutoff, I = p.InnerCutoff;
  k.cut2 = C * C;
  k.vdwcut2 = p.VdwCutoff * p.VdwCutoff;
  k.vdwcut_d = p.VdwCutoff;
  k.cut = (float)C;
  k.inner = (float)I;
  k.vdwcut = (float)p.VdwCutoff;
  k.vdwinner = (float)p.VdwInnerCutoff;
  // A zero switching width never switches (no pair has Inner < r <= Cutoff); keep
  // the device constants finite so the branch-free switch stays exactly 1.
  const double vw = p.VdwCutoff - p.VdwInnerCutoff;
  k.invw_vdw = vw > 0 ? (float)(1.0 / vw) : 0.0f;
  k.invw2_vdw4 = vw > 0 ? (float)(4.0 / (vw * vw)) : 0.0f;
  const double ew = C - I;
  k.invw_el = ew > 0 ? (float)(1.0 / ew) : 0.0f;
  k.invw2_el4 = ew > 0 ? (float)(4.0 / (ew * ew)) : 0.0f;
  // force-switch constants, nonbonded.cpp:620-636
  auto sqr = [](double v) { return v * v; };
  auto cube = [](double v) { return v * v * v; };
  const double sA = 1.0 / cube(sqr(C) - sqr(I));
  const double sB = -(cube(sqr(C)) - 3.0 * sqr(C) * sqr(C) * sqr(I));
  const double sC = 6.0 * sqr(C) * sqr(I);
  const double sD = -(sqr(C) + sqr(I));
  const double sE = 2.0 / 5.0;
  const double finner = sA * (sB * (1.0 / I) + sC * I + sD * cube(I) + sE * cube(I) * sqr(I));
  const double fcut = sA * (sB * (1.0 / C) + sC * C + sD * cube(C) + sE * cube(C) * sqr(C));
  const double eshift = (I < C) ? 1 / I + (finner - fcut) : 0.0;
  k.sA = (float)sA;
  k.sB = (float)sB;
  k.sC = (float)sC;
  k.sD = (float)sD;
  k.sE = (float)sE;
  k.fcut = (float)fcut;
  k.eshift = (float)eshift;
  k.rc2 = (float)(C * C);
  k.fs_c1 = (float)(sA * sB);
  k.fs_c2 = (float)(sA * sC);
  k.fs_c3 = (float)(sA * sD);
  k.fs_c4 = (float)(sA * sE);
  k.fs_k = (float)(C * C - 3.0 * I * I);
  k.fs_invw = (I < C) ? (float)(1.0 / (C * C - I * I)) : 0.0f;
  k.fs_x0 = (I < C) ? (float)(-(I * I) / (C * C - I * I)) : 0.0f;
  k.same_cut = (p.Cutoff == p.VdwCutoff) ? 1 : 0;
  k.rin2 = (float)(I * I);
  k.vdw14 = (float)p.Vdw14Scaling;
  k.elec14 = (float)p.Elec14Scaling;
  k.vdw_on = p.DoVdw ? 1 : 0;
  int mode = 1;  // dispatch as FF_NonBonded::calcForces, nonbonded.cpp:1228-1238
  if (p.EnergySwitch) mode = 3;
  if (p.ForceSwitch) mode = 4;
  if (!p.DoElec) mode = 0;
  k.elec_mode = mode;
  if (p.VdwCor) {
    const double R = p.VdwCorRadius;
    k.vdwcor_per_atom = -0.5 * p.VdwCorDensity * p.VdwCorEpsilon * (8.0 / 3.0) * Consts::PI * sqr(R) *
                        sqr(R) * sqr(R) / cube(p.VdwCorCutoff);  // kcal/mol
  }
  k.d.vdw14 = p.Vdw14Scaling;
  k.d.elec14 = p.Elec14Scaling;
  k.d.vdwinner = p.VdwInnerCutoff;
  k.d.invw_vdw = vw > 0 ? 1.0 / vw : 0.0;
  k.d.invw2_vdw4 = vw > 0 ? 4.0 / (vw * vw) : 0.0;
  k.d.inner = I;
  k.d.invw_el = ew > 0 ? 1.0 / ew : 0.0;
  k.d.invw2_el4 = ew > 0 ? 4.0 / (ew * ew) : 0.0;
  k.d.fcut = fcut;
  k.d.eshift = eshift;
  k.d.fs_c1 = sA * sB;
  k.d.fs_c2 = sA * sC;
  k.d.fs_c3 = sA * sD;
  k.d.fs_c4 = sA * sE;
  k.d.fs_invw = (I < C) ? 1.0 / (C * C - I * I) : 0.0;
  k.d.fs_x0 = (I < C) ? -(I * I) / (C * C - I * I) : 0.0;
  nbk = k;
  // per-atom parameters in kernel units: charge * sqrt(econv/Dielectric), sqrt(eps[kcal/mol])
  std::vector<float> q(n), r(n), e(n);
  std::vector<float4> lo(n);
  const double qs = std::sqrt(Consts::econv() / p.Dielectric);
  const double es = 1.0 / std::sqrt(Consts::kcal_to_J());
  for (int i = 0; i < n; i++) {
    const double qi = h_charge[i] * qs, ei = h_epsilon[i] * es;
    q[i] = (float)qi;
    r[i] = (float)h_radius[i];
    e[i] = (float)ei;
    lo[i] = make_float4((float)(qi - q[i]), (float)(h_radius[i] - r[i]), (float)(ei - e[i]), 0.0f);
  }
  q_scaled.upload(q, stream);
  lj_r.upload(r, stream);
  lj_e.upload(e, stream);
  prm_lo.upload(lo, stream);
  have_nb = true;
  list_valid = false;
}

void Engine::begin_evaluation(bool nonbonded, double *eo, bool opened, bool gb_next) {
  const int T = 256;
  fbx.resize(n);
  fby.resize(n);
  fbz.resize(n);
  e_out.resize(24);
  if (!eo) eo = e_out.p;
  // a pending MD step's energy sums run in this kernel; e_out then keeps its
  // values (every slot a component fills is assigned by the sums)
  SumList L{};
  const int zero_e = fused_pending ? 0 : 1;
  if (fused_pending) {
    L = fused_sums;
    fused_pending = false;
  }
  gb_sums = SumList{};
  if (!nonbonded && gb_next) {  // the sums run in k_gb_open
    gb_sums = L;
    L = SumList{};
  }
  if (!nonbonded && opened) {  // the previous step's integrator cleared the accumulators
    require(!zero_e, "an opened evaluation keeps its energy slots");
    return;
  }
  if (!nonbonded) {
    hipLaunchKernelGGL(k_begin_nb, dim3((std::max(n, 24) + T - 1) / T), dim3(T), 0, stream, 0, n, n_clusters_d.p,
                       nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, nullptr, nullptr,
                       nullptr, fbx.p, fby.p, fbz.p, eo, 24, zero_e, L);
    return;
  }
  require(list_valid, "neighbour list not built");
  size_eval_buffers();
  dmax_cur ^= 1;
  const int nslots = max_clusters * kClusterSize;
  const int m = std::max(std::max(nslots, n), 24);
  // the pending sums run in the nonbonded kernel's first workgroup instead
  nb_sums = L;
  nb_sums_pending = L.n > 0 || L.record;
  if (opened) {  // the previous step's integrator did this kernel's work
    require(!zero_e, "an opened evaluation keeps its energy slots");
    return;
  }
  hipLaunchKernelGGL(k_begin_nb, dim3((m + T - 1) / T), dim3(T), 0, stream, nslots, n, n_clusters_d.p, slot_orig.p,
                     x.p, y.p, z.p, spos.p, spos32.p, pref.p, prune_dmax.p, dmax_cur, nbx.p, nby.p, nbz.p, fbx.p, fby.p, fbz.p,
                     eo, 24, zero_e, SumList{});
}

// Every buffer an evaluation with the nonbonded term writes, sized for the
// current list (a no-op when they are large enough): called at each list build,
// so that evaluations between builds allocate nothing.
void Engine::size_eval_buffers() {
  fbx.resize(n);
  fby.resize(n);
  fbz.resize(n);
  e_out.resize(24);
  const int nslots = max_clusters * kClusterSize;
  spos.resize(nslots);
  spos32.resize(nslots);
  pref.resize(nslots);
  const size_t ndm = 2 * kDmaxSpread * kDmaxStride;
  if (prune_dmax.n < ndm) {
    prune_dmax.resize(ndm);
    PDGPU_HIP(hipMemsetAsync(prune_dmax.p, 0, ndm * sizeof(unsigned), stream));
  }
  pentries.resize((size_t)max_clusters * entry_capacity);
  pcount.resize(max_clusters);
  pcount_nolj.resize(max_clusters);
  // Few groups leave most of the 256 CUs idle and every wave with one long chain of
  // rounds, so up to 384 groups two waves share a cluster, four atoms each in FP64
  // (k_nonbonded's FINE: the FP64 units would idle as well), and each group has two
  // workgroups with every other round, up to 128 groups four.  An MD step of water in
  // us, FP32 with one workgroup a group | FINE with 2 | 3 | 4 | 6: 1,536 atoms (80
  // groups) 49 | 41 | 38 | 37 | 39; 3,072 (168) 50 | 42 | 42 | 43 | 47; 6,144 (344)
  // 51 | 49 | 51 | 55 | 61; 12,288 (536) 55 | 62 | 68 | 73 | 84.  More workgroups repeat
  // the prologue and the flush of the j forces; a filled chip is bound by issue.
  nb_share = max_groups <= 384 ? 2 : 1;
  nb_parts = max_groups <= 128 ? 4 : max_groups <= 384 ? 2 : 1;
  const size_t np = (size_t)max_groups * nb_parts * 4;
  if (fused_pending && e_partial.n < np) run_fused_sums();  // they read the arrays that grow here
  e_partial.resize(np);
  e_partial_b.resize(np);
}

// Per-slot parameters and accumulators; called once per list rebuild.
void Engine::prepare_slots() {
  const int nslots = max_clusters * kClusterSize;
  sprm.resize(nslots);  // filled by the column sort
  sprm_lo.resize(nslots);
  nbx.resize(nslots);
  nby.resize(nslots);
  nbz.resize(nslots);
}

void Engine::launch_nonbonded(double *energy_out, bool forces, double *partial, double *bonded_out) {
  require(have_nb, "nonbonded component not set up");
  require(list_valid, "neighbour list not built");
  {
    ScopedTimer t(*this, "prune");
    const double rk = std::max(nb.Cutoff, nb.VdwCutoff) + prune_margin;
    const GroupOrderArgs G{order_due ? 1 : 0, max_groups, nb_per_cap, n_groups_d.p, grp_work.p, grp_order.p};
    const int pblocks = (max_clusters + kPruneWaves - 1) / kPruneWaves + (order_due ? 1 : 0);
    order_due = false;
    hipLaunchKernelGGL(k_prune, dim3(pblocks), dim3(64 * kPruneWaves), 0,
                       stream, n_clusters_d.p,
                       periodic ? box[0] : 0.0, periodic ? box[1] : 0.0, periodic ? box[2] : 0.0,
                       (float)(rk * rk), (float)(prune_margin - 1e-3), prune_forced ? 1 : 0, prune_dmax.p + dmax_cur * kDmaxSpread * kDmaxStride, spos.p,
                       spos32.p, entries.p, cl_entry_count.p, (int)entry_capacity, pentries.p, pcount.p,
                       pcount_nolj.p, pref.p, G);
    prune_forced = false;
  }
  const int sel = e_partial_sel;
  if (!partial) {  // alternate arrays: a previous step's sums may still read the other
    partial = e_partial_sel ? e_partial_b.p : e_partial.p;
    e_partial_sel ^= 1;
  }
  const SumList L = nb_sums_pending ? nb_sums : SumList{};
  nb_sums_pending = false;
  double *bp = nullptr;
  const int nbb = bonded_blocks(nbonds, nangles, ntors);
  if (bonded_out) {
    e_partial_bonded.resize((size_t)nbb * 8);  // alternating halves, as above
    bp = e_partial_bonded.p + (size_t)sel * nbb * 4;
  }
  nbk.fine = nb_share > 1;
  const bool v = nbk.vdw_on != 0;
  {
    ScopedTimer t(*this, "nonbonded");
    switch (nbk.elec_mode) {
      case 0: launch_mode<EL_NONE>(*this, v, forces, partial, L, bp); break;
      case 1: launch_mode<EL_PLAIN>(*this, v, forces, partial, L, bp); break;
      case 3: launch_mode<EL_ESWITCH>(*this, v, forces, partial, L, bp); break;
      default: launch_mode<EL_FSWITCH>(*this, v, forces, partial, L, bp); break;
    }
  }
  PDGPU_HIP(hipGetLastError());
  defer_sum4(partial, max_groups * nb_parts, energy_out);
  if (bonded_out) defer_sum4(bp, nbb, bonded_out);
}

}  // namespace pdgpu
