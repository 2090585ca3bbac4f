// k_partial.hip -- FF_NonBonded::calcEnergies with UsePartialRecalc on the device
// (nonbonded.cpp:1154-1181 and FF_NonBonded_CalcEnergies_Update_T, 76-386): the
// nonbonded energy after a Monte Carlo move from the energy before it, by
// re-evaluating only the pairs that touch an atom whose position changed.
//
// PD keeps the coordinates of its last energy evaluation (WorkSpace::old), lists
// the atoms whose position differs, and for each of them takes every non-bonded
// or 1-4 partner: the pair's energy at the old positions is subtracted and the
// energy at the new ones added (a pair of two moved atoms once).  After a list
// rebuild (a new full-update count) it evaluates the whole energy instead.
//
// Here the moved atoms are found and listed in index order by one workgroup; a
// grid of (moved atom, block of 256 partners) then evaluates each pair in FP64
// with PD's energy expressions at both positions, the partner's bond order
// looked up as the list builder assigns it, and the per-block differences are
// summed in a fixed order.  The pair set is every partner within Cutoff (minimum
// image in a PeriodicBox), which is PD's list-based set while the list is valid.  Past kPartialMax moved atoms a full evaluation is cheaper and is
// taken; its result is the same energy.
#include "engine.hpp"

#include <cmath>

namespace pdgpu {

namespace {

constexpr int kPartialMax = 256;  // moved atoms handled by the pair update
constexpr int kCompactThreads = 1024;

struct PartialArgs {
  int n;
  int periodic;
  double L[3], half[3];
  double cut, inner, vdwcut, vdwinner;
  double invw, vinvw;
  double econv, invdiel;
  double vdw14, elec14;
  int vdw_on, elec_mode;  // 0 none, 1 plain, 3 energy switch, 4 force switch
  double sA, sB, sC, sD, sE, fcut, eshift;
  int mid;
};

// Moved atoms (any coordinate differs from the snapshot) listed in index order.
__global__ __launch_bounds__(kCompactThreads) void k_pr_compact(int n, const double *__restrict__ x,
                                                                const double *__restrict__ y,
                                                                const double *__restrict__ z,
                                                                const double *__restrict__ ox,
                                                                const double *__restrict__ oy,
                                                                const double *__restrict__ oz,
                                                                int *__restrict__ moved, int *__restrict__ count) {
  constexpr int W = kCompactThreads / 64;
  __shared__ int wcount[W];
  __shared__ int base;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (threadIdx.x == 0) base = 0;
  __syncthreads();
  for (int i0 = 0; i0 < n; i0 += kCompactThreads) {
    const int i = i0 + (int)threadIdx.x;
    const bool m = i < n && !(x[i] == ox[i] && y[i] == oy[i] && z[i] == oz[i]);
    const unsigned long long b = __ballot(m);
    if (lane == 0) wcount[w] = __popcll(b);
    __syncthreads();
    int off = base;
    for (int k = 0; k < w; k++) off += wcount[k];
    if (m) moved[off + __popcll(b & ((1ull << lane) - 1ull))] = i;
    __syncthreads();
    if (threadIdx.x == 0) {
      int t = 0;
      for (int k = 0; k < W; k++) t += wcount[k];
      base += t;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) count[0] = base;
}

// BondOrder of (a, b) as the list builder assigns it (band matrix, then the
// off-diagonal partners; the last one of a pair wins).
__device__ __forceinline__ int pr_bond_order(int a, int b, int mid, const int8_t *__restrict__ band,
                                             const int *__restrict__ sp_off, const int *__restrict__ sp_part,
                                             const int *__restrict__ sp_ord) {
  const int hi = max(a, b), lo = min(a, b);
  int bo = 7;
  if (hi - lo < mid) bo = band[(long)lo * mid + (hi - lo - 1)];
  for (int k = sp_off[lo]; k < sp_off[lo + 1]; k++)
    if (sp_part[k] == hi) bo = sp_ord[k];
  return bo & 7;
}

// One pair's vdW and Coulomb energies (J) as FF_NonBonded_CalcEnergies_Update_T
// computes them (nonbonded.cpp:297-371), for the displacement d = p_j - p_i.
__device__ void pr_pair_energy(const PartialArgs &A, double dx, double dy, double dz, double ri, double ei,
                               double qi, double rj, double ej, double qj, double s_vdw, double s_elec, double &ev,
                               double &ee) {
#pragma clang fp contract(off)
  ev = 0.0;
  ee = 0.0;
  if (A.periodic) {  // the minimum image, by PD's wrapping loops
    for (int it = 0; it < 8 && dx > A.half[0]; it++) dx -= A.L[0];
    for (int it = 0; it < 8 && dx < -A.half[0]; it++) dx += A.L[0];
    for (int it = 0; it < 8 && dy > A.half[1]; it++) dy -= A.L[1];
    for (int it = 0; it < 8 && dy < -A.half[1]; it++) dy += A.L[1];
    for (int it = 0; it < 8 && dz > A.half[2]; it++) dz -= A.L[2];
    for (int it = 0; it < 8 && dz < -A.half[2]; it++) dz += A.L[2];
  }
  const double r2 = dx * dx + dy * dy + dz * dz;
  // the full evaluation's pair set (fast2 skips r^2 > Cutoff^2, nonbonded.cpp:722);
  // PD's InfiniteSpace update omits this test, which differs only for VdwCutoff > Cutoff
  if (r2 > A.cut * A.cut) return;
  const double r = sqrt(r2);
  const double ir = 1.0 / r;
  if (A.vdw_on && r < A.vdwcut) {
    const double eps = s_vdw * ei * ej;
    double B = (ri + rj) * ir;
    B = B * B;
    B *= B * B;
    const double Av = B * B;
    ev = (2.0 * eps) * (0.5 * Av - B);
    if (r > A.vdwinner) {
      double S = 1.0 - (A.vinvw * (r - A.vdwinner)) * (A.vinvw * (r - A.vdwinner));
      S = S * S;
      ev *= S;
    }
  }
  if (A.elec_mode != 0 && r < A.cut) {
    if (A.elec_mode == 3) {
      ee = A.econv * A.invdiel * s_elec * (qi * qj) * ir;
      if (r > A.inner) {
        double S = 1.0 - (A.invw * (r - A.inner)) * (A.invw * (r - A.inner));
        S = S * S;
        ee *= S;
      }
    } else if (A.elec_mode == 4) {
      ee = A.econv * A.invdiel * s_elec * (qi * qj);
      if (r > A.inner)
        ee *= -(A.sA * r * (A.sB * (ir * ir) + A.sC + A.sD * r2 + A.sE * (r2 * r2)) - A.fcut);
      else
        ee *= (ir - A.eshift);
    } else {
      ee = A.econv * A.invdiel * s_elec * (qi * qj) * ir;
    }
  }
}

// Block (a, b): moved atom moved[a] against partners b*256 .. b*256+255; writes
// the block's sum of (new - old) vdW and Coulomb energies.
__global__ __launch_bounds__(256) void k_pr_update(PartialArgs A, const int *__restrict__ moved,
                                                   const double *__restrict__ x, const double *__restrict__ y,
                                                   const double *__restrict__ z, const double *__restrict__ ox,
                                                   const double *__restrict__ oy, const double *__restrict__ oz,
                                                   const double *__restrict__ rad, const double *__restrict__ eps,
                                                   const double *__restrict__ chg, const int8_t *__restrict__ band,
                                                   const int *__restrict__ sp_off, const int *__restrict__ sp_part,
                                                   const int *__restrict__ sp_ord, double *__restrict__ part) {
#pragma clang fp contract(off)
  __shared__ double s[2][4];
  const int i = moved[blockIdx.x];
  const int j = (int)blockIdx.y * 256 + (int)threadIdx.x;
  double dv = 0.0, de = 0.0;
  if (j < A.n && j != i) {
    // a pair of two moved atoms counts once: from its lower moved atom
    const bool j_moved = !(x[j] == ox[j] && y[j] == oy[j] && z[j] == oz[j]);
    if (!(j_moved && j < i)) {
      const int bo = pr_bond_order(i, j, A.mid, band, sp_off, sp_part, sp_ord);
      if (bo >= 3) {  // non-bonded and 1-4 partners
        const double sv = bo == 3 ? A.vdw14 : 1.0, se = bo == 3 ? A.elec14 : 1.0;
        double ev0, ee0, ev1, ee1;
        pr_pair_energy(A, ox[j] - ox[i], oy[j] - oy[i], oz[j] - oz[i], rad[i], eps[i], chg[i], rad[j], eps[j],
                       chg[j], sv, se, ev0, ee0);
        pr_pair_energy(A, x[j] - x[i], y[j] - y[i], z[j] - z[i], rad[i], eps[i], chg[i], rad[j], eps[j], chg[j],
                       sv, se, ev1, ee1);
        dv = ev1 - ev0;
        de = ee1 - ee0;
      }
    }
  }
  dv = wave_sum(dv);
  de = wave_sum(de);
  if ((threadIdx.x & 63) == 0) {
    s[0][threadIdx.x >> 6] = dv;
    s[1][threadIdx.x >> 6] = de;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const double t = ((s[threadIdx.x][0] + s[threadIdx.x][1]) + s[threadIdx.x][2]) + s[threadIdx.x][3];
    part[2 * ((size_t)blockIdx.x * gridDim.y + blockIdx.y) + threadIdx.x] = t;
  }
}

// The first workgroup: the block sums in a fixed order (thread t: blocks t, t+256,
// ...; then the threads in order), stored to out (pinned host memory).  The others:
// the snapshot takes the current positions for the next update
// (getWSpace().old = getWSpace().cur).
__global__ __launch_bounds__(256) void k_pr_finish(int nparts, const double *__restrict__ part,
                                                   double *__restrict__ out, int n, const double *__restrict__ x,
                                                   const double *__restrict__ y, const double *__restrict__ z,
                                                   double *__restrict__ ox, double *__restrict__ oy,
                                                   double *__restrict__ oz) {
  __shared__ double s[2][256];
  if (blockIdx.x > 0) {
    const int i = (blockIdx.x - 1) * 256 + threadIdx.x;
    if (i < n) {
      ox[i] = x[i];
      oy[i] = y[i];
      oz[i] = z[i];
    }
    return;
  }
  double v = 0.0, e = 0.0;
  for (int k = threadIdx.x; k < nparts; k += 256) {
    v += part[2 * k];
    e += part[2 * k + 1];
  }
  s[0][threadIdx.x] = v;
  s[1][threadIdx.x] = e;
  __syncthreads();
  if (threadIdx.x < 2) {
    double t = 0.0;
    for (int k = 0; k < 256; k++) t += s[threadIdx.x][k];
    out[threadIdx.x] = t;
  }
}

__global__ void k_pr_snapshot(int n, const double *__restrict__ x, const double *__restrict__ y,
                              const double *__restrict__ z, double *__restrict__ ox, double *__restrict__ oy,
                              double *__restrict__ oz) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  ox[i] = x[i];
  oy[i] = y[i];
  oz[i] = z[i];
}

}  // namespace

void Engine::energy_update(uint32_t components, pdgpu_energies *out) {
  require(components == PDGPU_NONBONDED,
          "pdgpu_energy_update evaluates FF_NonBonded alone (other components: pdgpu_compute)");
  require(have_nb, "nonbonded component not set up");
  require(have_positions, "positions not set");
  const int T = 256;
  const int grid = (n + T - 1) / T;
  pr_x.resize(n);
  pr_y.resize(n);
  pr_z.resize(n);
  pr_moved.resize(n);
  // the count of moved atoms and the update's sums come back in pinned memory
  int *h_count = reinterpret_cast<int *>(h_eout);
  double *h_sum = h_eout + 1;
  // a list rebuild since the snapshot forces a full evaluation (nonbonded.cpp:1157-1162)
  const bool full = !pr_valid || !list_valid || pr_update_count != full_update_count;
  int m = 0;
  if (!full) {
    hipLaunchKernelGGL(k_pr_compact, dim3(1), dim3(kCompactThreads), 0, stream, n, x.p, y.p, z.p, pr_x.p, pr_y.p,
                       pr_z.p, pr_moved.p, h_count);
    PDGPU_HIP(hipGetLastError());
    sync();
    m = *h_count;
  }
  if (full || m > kPartialMax) {
    pr_rad.upload(h_radius, stream);
    pr_eps.upload(h_epsilon, stream);
    pr_chg.upload(h_charge, stream);
    evaluate(PDGPU_NONBONDED | PDGPU_ENERGY_ONLY, 0, true);
    pdgpu_energies e{};
    energies_to_host(PDGPU_NONBONDED, &e);
    pr_vdw = e.epot_vdw;
    pr_elec = e.epot_elec;
    pr_update_count = full_update_count;
    pr_valid = true;
    hipLaunchKernelGGL(k_pr_snapshot, dim3(grid), dim3(T), 0, stream, n, x.p, y.p, z.p, pr_x.p, pr_y.p, pr_z.p);
    PDGPU_HIP(hipGetLastError());
    sync();
  } else if (m > 0) {
    PartialArgs A{};
    A.n = n;
    A.periodic = periodic ? 1 : 0;
    for (int d = 0; d < 3; d++) {
      A.L[d] = periodic ? box[d] : 0.0;
      A.half[d] = periodic ? box[d] / 2.0 : 0.0;
    }
    A.cut = nb.Cutoff;
    A.inner = nb.InnerCutoff;
    A.vdwcut = nb.VdwCutoff;
    A.vdwinner = nb.VdwInnerCutoff;
    A.invw = 1.0 / (nb.Cutoff - nb.InnerCutoff);
    A.vinvw = 1.0 / (nb.VdwCutoff - nb.VdwInnerCutoff);
    A.econv = Consts::econv_joule();
    A.invdiel = 1.0 / nb.Dielectric;
    A.vdw14 = nb.Vdw14Scaling;
    A.elec14 = nb.Elec14Scaling;
    A.vdw_on = nb.DoVdw ? 1 : 0;
    A.elec_mode = !nb.DoElec ? 0 : (nb.ForceSwitch ? 4 : (nb.EnergySwitch ? 3 : 1));
    const double C = nb.Cutoff, I = nb.InnerCutoff;
    A.sA = 1.0 / std::pow(C * C - I * I, 3.0);
    A.sB = -(std::pow(C * C, 3.0) - 3.0 * (C * C) * (C * C) * (I * I));
    A.sC = 6.0 * (C * C) * (I * I);
    A.sD = -(C * C + I * I);
    A.sE = 2.0 / 5.0;
    const double fin = A.sA * (A.sB * (1.0 / I) + A.sC * I + A.sD * (I * I * I) + A.sE * (I * I * I) * (I * I));
    A.fcut = A.sA * (A.sB * (1.0 / C) + A.sC * C + A.sD * (C * C * C) + A.sE * (C * C * C) * (C * C));
    A.eshift = I < C ? 1 / I + (fin - A.fcut) : 0.0;
    A.mid = mid;
    const int nb_blocks = grid;
    pr_part.resize((size_t)m * nb_blocks * 2);
    hipLaunchKernelGGL(k_pr_update, dim3(m, nb_blocks), dim3(256), 0, stream, A, pr_moved.p, x.p, y.p, z.p, pr_x.p,
                       pr_y.p, pr_z.p, pr_rad.p, pr_eps.p, pr_chg.p, band.p, sp_off.p, sp_part.p, sp_ord.p,
                       pr_part.p);
    hipLaunchKernelGGL(k_pr_finish, dim3(1 + grid), dim3(256), 0, stream, m * nb_blocks, pr_part.p, h_sum, n, x.p,
                       y.p, z.p, pr_x.p, pr_y.p, pr_z.p);
    PDGPU_HIP(hipGetLastError());
    sync();
    pr_vdw += h_sum[0];
    pr_elec += h_sum[1];
  }
  pdgpu_energies e{};
  e.epot_vdw = pr_vdw;
  e.epot_elec = pr_elec;
  e.epot = pr_vdw + pr_elec;
  *out = e;
}

}  // namespace pdgpu
