// k_bonded.hip -- FF_Bonded bond, angle and torsion forces on the device (FP64).
//
// One thread per term, PD's formulas (ffbonded.cpp:945-992 bonds, 1054-1177
// angles, 1274-1512 dihedrals) in kcal/mol and Angstrom.  Forces go to the
// original-order 64-bit fixed-point accumulators, energies to per-block FP64
// partials reduced in a fixed order.  The terms of a block of 256 (never
// mixing kinds) usually touch a short run of consecutive atoms; the block then
// sums its forces in an LDS window over that run and adds the window to global
// memory once, with consecutive threads on consecutive atoms: global atomics
// run at a bounded rate per lane operation on this GPU and scattered ones far
// below it, so this replaces up to 12 scattered atomics per term by a few
// coalesced ones per atom.
#include "bonded_dev.hpp"

#include <algorithm>
#include <climits>

namespace pdgpu {

namespace {

__global__ __launch_bounds__(256) void k_bonded(BondedArrays B, const double *__restrict__ x,
                                                const double *__restrict__ y, const double *__restrict__ z,
                                                long long *__restrict__ fx, long long *__restrict__ fy,
                                                long long *__restrict__ fz, double *__restrict__ partial,
                                                double *__restrict__ eterm) {
  __shared__ long long acc[3 * kBondedWindow];
  bonded_block((int)blockIdx.x, B, x, y, z, fx, fy, fz, partial, eterm, acc);
}

}  // namespace

int bonded_blocks(int nb, int na, int nt) {
  return std::max(1, (nb + 255) / 256 + (na + 255) / 256 + (nt + 255) / 256);
}

std::vector<int2> bonded_windows(int nb, const int *bi, const int *bj, int na, const int *ai, const int *aa,
                                 const int *aj, int nt, const int *ti, const int *ta, const int *tb, const int *tj) {
  std::vector<int2> w;
  auto kind = [&](int cnt, std::initializer_list<const int *> idx) {
    for (int b0 = 0; b0 < cnt; b0 += 256) {
      int lo = INT32_MAX, hi = -1;
      for (int t = b0; t < std::min(cnt, b0 + 256); t++)
        for (const int *a : idx) {
          lo = std::min(lo, a[t]);
          hi = std::max(hi, a[t]);
        }
      w.push_back(hi - lo + 1 <= kBondedWindow ? make_int2(lo, hi - lo + 1) : make_int2(0, 0));
    }
  };
  kind(nb, {bi, bj});
  kind(na, {ai, aa, aj});
  kind(nt, {ti, ta, tb, tj});
  if (w.empty()) w.push_back(make_int2(0, 0));
  return w;
}

void launch_bonded_kernel(hipStream_t s, const BondedArrays &B, const double *x, const double *y,
                          const double *z, long long *fx, long long *fy, long long *fz, double *partial,
                          double *eterm) {
  const int grid = bonded_blocks(B.nb, B.na, B.nt);
  hipLaunchKernelGGL(k_bonded, dim3(grid), dim3(256), 0, s, B, x, y, z, fx, fy, fz, partial, eterm);
}

BondedArrays Engine::bonded_arrays() const {
  return BondedArrays{nbonds, nangles, ntors, b_i.p, b_j.p, b_l.p, b_k.p, a_i.p, a_a.p, a_j.p, a_t0.p, a_k.p,
                      t_i.p, t_a.p, t_b.p, t_j.p, t_terms.p, t_vn.p, t_nn.p, t_gamma.p, b_win.p};
}

void Engine::launch_bonded(double *energy_out, double *partial) {
  const int grid = bonded_blocks(nbonds, nangles, ntors);
  if (!partial) {
    e_partial_bonded.resize((size_t)grid * 4);
    partial = e_partial_bonded.p;
  }
  launch_bonded_kernel(stream, bonded_arrays(), x.p, y.p, z.p, fbx.p, fby.p, fbz.p, partial, nullptr);
  PDGPU_HIP(hipGetLastError());
  defer_sum4(partial, grid, energy_out);
}

}  // namespace pdgpu
