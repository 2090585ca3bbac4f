// k_lcpo.hip -- FF_SASA_LCPO (LCPO solvent-accessible surface) on the device.
//
// Restates FF_SASA_LCPO::calcLCPOSasaForces (lcpo.cpp:643-962), the linear
// combination of pairwise overlaps of Weiser, Shenkin & Still:
//   SASA_i = P1 S_i + P2 sum_j A_ij + P3 sum_j sum_k A_jk + P4 sum_j A_ij sum_k A_jk
// over the overlap neighbours j of i and the neighbours k of j that also
// overlap i, with S_i = 4 pi R_i^2, R = LCPO radius + 1.4 A, and the energy
// sum_i sigma_i SASA_i (lcpo.cpp:63).  Three kernels:
//   k_lcpo_lists  one wavefront per atom over the 64-atom tiles near it: the
//                 overlap partners (d < R_i + R_j, hydrogens excluded) in
//                 ascending index order, at most 80 (Nlistmax, lcpo.h:24) --
//                 the order and truncation PD's fill loop produces
//                 (lcpo.cpp:713-767); for the energy path also, one lane per
//                 partner, the overlap A_ij = 2 pi R_i (R_i - d/2 - (R_i^2 - R_j^2) / 2d);
//   k_lcpo_sasa   one wavefront per atom: SASA_i and the derivative that PD
//                 collects on atom i (its own self terms plus the derivatives
//                 of its neighbours' SASA with respect to x_i), clamped to zero
//                 with the SASA when SASA_i < 0 (lcpo.cpp:940-944);
//   k_lcpo_apply  every step: adds the stored derivative to the force
//                 accumulators and writes sigma_i SASA_i.
// PD recomputes only every UpdateSasa steps and re-applies the stored forces in
// between (lcpo.cpp:196-201, 659-677); the first two kernels return at once on
// the other steps (the step is read on the device, so a captured graph replays
// correctly).  Overlap partners are searched over all atoms of the atom's
// system, which is PD's neighbour list whenever that list holds every pair
// within R_i + R_j (the all-pairs GB/SA setting, or any list of at least 7 A,
// lcpo.cpp:37).  Everything is FP64 in PD's expression order, so the SASA and
// forces agree with the CPU arithmetic to FP64 rounding (the
// sums are taken in a different order).
#include "engine.hpp"

#include <algorithm>
#include <climits>
#include <cmath>

namespace pdgpu {

namespace {

// EONLY: the overlap lists of calcLCPOSasaEnergies (lcpo.cpp:469-520): the test
// on the distance itself and sphereSurfaceOverlap clamped at zero.
// One wave per atom i at a time (kListWaves waves per workgroup, each striding over the atoms).  The lanes first test
// 64 tiles of i's system at a time (64 consecutive atoms each, by the box of
// their used atoms) against R_i + max R; then, tile by tile in ascending order,
// each near tile's 64 atoms one per lane, and a ballot places the partners in
// index order, so each list comes out ascending and the first kLcpoMax are
// kept, as PD's fill loop does.  A list that is cut at kLcpoMax, or has a partner at
// exactly R_i + R_j (no partner, but still inside the test of PD's inner loop), is
// flagged (kListCut) for k_lcpo_sasa.  EONLY: the overlaps follow, one lane per partner.
constexpr int kListWaves = 4;
constexpr int kListCut = 0x100;  // in nl_cnt, above the count
// workgroups of k_lcpo_lists at most (each wave walks atoms wave, + 4 * grid, ...):
// the launch returns at once on the steps that re-apply the stored forces, and
// the cost of that empty launch grows with its workgroup count (16 us for the
// 68,864 workgroups of one wave per atom on the 275k-atom chain batch)
constexpr int kListGrid = 16384;
template <bool EONLY>
__global__ __launch_bounds__(64 * kListWaves) void k_lcpo_lists(
    int n, const int *__restrict__ atom_sys, const int *__restrict__ sys_first, const int *__restrict__ sys_count,
    const double4 *__restrict__ pr, const double *__restrict__ tile_box, double max_R,
    int *__restrict__ nl_cnt,
    int *__restrict__ nl_idx, double *__restrict__ nl_s) {
#pragma clang fp contract(off)
  __shared__ int s_list[kListWaves][kLcpoMax];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // whole waves; no barrier follows
  for (int i = blockIdx.x * kListWaves + wave; i < n; i += gridDim.x * kListWaves) {
    const double4 pi = pr[i];
    if (!(pi.w > 0.0)) {  // R < 0: an atom LCPO does not use
      if (lane == 0) nl_cnt[i] = 0;
      continue;
    }
    const int sy = atom_sys[i];
    const int first = sys_first[sy], end = first + sys_count[sy];
    const double ri = pi.w;
    // a partner j has d < R_i + R_j <= R_i + max R, so its tile's box lies within that
    // (the box's distance never exceeds the atom's: rounding is monotonic); the
    // factor keeps the test on the safe side of the last bit
    const double reach = (ri + max_R) * (1.0 + 1e-12);
    const unsigned long long below = (1ull << lane) - 1ull;
    int *my = s_list[wave];
    int cnt = 0, cut = 0;
    const int tfirst = first / 64, tlast = (end - 1) / 64;
    // one past the last partner that is kept, to know whether any is dropped
    for (int t0 = tfirst; t0 <= tlast && cnt <= kLcpoMax; t0 += 64) {
      bool near = false;
      const int t = t0 + lane;
      if (t <= tlast) {
        const double *bx = tile_box + 6 * (size_t)t;
        const double gx = fmax(0.0, fmax(bx[0] - pi.x, pi.x - bx[3]));
        const double gy = fmax(0.0, fmax(bx[1] - pi.y, pi.y - bx[4]));
        const double gz = fmax(0.0, fmax(bx[2] - pi.z, pi.z - bx[5]));
        near = gx * gx + gy * gy + gz * gz <= reach * reach;
      }
      unsigned long long nb = __ballot(near);
      while (nb != 0ull && cnt <= kLcpoMax) {
        const int tt = t0 + __ffsll((long long)nb) - 1;
        nb &= nb - 1ull;
        const int j = tt * 64 + lane;
        bool ok = false, edge = false;
        if (j >= first && j < end && j != i) {
          const double4 pj = pr[j];
          if (pj.w > 0.0) {
            const double g = pi.x - pj.x, h = pi.y - pj.y, k = pi.z - pj.z;
            const double d2 = g * g + h * h + k * k;
            const double rj = pj.w;
            ok = EONLY ? sqrt(d2) < (ri + rj) : d2 < (ri + rj) * (ri + rj);
            edge = !EONLY && d2 == (ri + rj) * (ri + rj);
          }
        }
        if (__ballot(edge) != 0ull) cut = kListCut;
        const unsigned long long b = __ballot(ok);
        const int pos = cnt + __popcll(b & below);
        if (ok && pos < kLcpoMax) {
          my[pos] = j;
          nl_idx[(size_t)i * kLcpoMax + pos] = j;
        }
        cnt += __popcll(b);
      }
    }
    if (cnt > kLcpoMax) cut = kListCut;
    cnt = min(cnt, kLcpoMax);
    if (lane == 0) nl_cnt[i] = EONLY ? cnt : cnt | cut;
    if (!EONLY) continue;
    // the list is read back by other lanes of the same wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // the overlaps: same expressions as PD, in its order
    const double TwoPI = 2.0 * Consts::PI;
    for (int c = lane; c < cnt; c += 64) {
      const int j = my[c];
      const double4 pj = pr[j];
      const double g = pi.x - pj.x, h = pi.y - pj.y, k = pi.z - pj.z;
      const double d2 = g * g + h * h + k * k;
      const double rj = pj.w;
      const double d = sqrt(d2);
      // sphereSurfaceOverlap (maths.cpp:120-123), negative overlaps set to 0
      double sij = TwoPI * ri * (ri - d / 2.0 - (ri * ri - rj * rj) / (2.0 * d));
      if (sij < 0) sij = 0;
      nl_s[(size_t)i * kLcpoMax + c] = sij;
    }
    // the next atom's list overwrites this one after every lane has read it
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// Packs position and LCPO radius per atom (R < 0 for atoms LCPO does not use),
// and the box of each 64-atom tile's used atoms (lo xyz, hi xyz; empty when
// none is used).  Blocks are whole waves, one tile each.
__global__ void k_lcpo_pack(int n, const double *__restrict__ x, const double *__restrict__ y,
                            const double *__restrict__ z, const int8_t *__restrict__ use,
                            const double *__restrict__ R, double4 *__restrict__ pr, double *__restrict__ tile_box) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  bool act = false;
  double p[3] = {0.0, 0.0, 0.0};
  if (i < n) {
    p[0] = x[i];
    p[1] = y[i];
    p[2] = z[i];
    act = use[i] != 0;
    pr[i] = make_double4(p[0], p[1], p[2], act ? R[i] : -1.0);
  }
  double lo[3], hi[3];
  for (int d = 0; d < 3; d++) {
    lo[d] = wave_min(act ? p[d] : 1e300);
    hi[d] = wave_max(act ? p[d] : -1e300);
  }
  const int t = i >> 6;
  if ((threadIdx.x & 63) == 0 && t * 64 < n)
    for (int d = 0; d < 3; d++) {
      tile_box[6 * (size_t)t + d] = lo[d];
      tile_box[6 * (size_t)t + 3 + d] = hi[d];
    }
}

// The SASA of atom i and the derivative PD collects on it (lcpo.cpp:786-948),
// one wavefront per atom.  PD's loops over the overlap neighbours j of i and
// the neighbours k of j are rearranged as one flat sum over the (j, k) pairs:
// every k-term enters the derivative linearly, with weights that depend on j
// alone (P3_j sigma_j, P4_j sigma_j, the overlap s_ji, the pair derivative of
// s_ji).
//
// The k that count are neighbours of j that overlap i: when the lists of i and of its
// neighbours are whole (kListCut unset), that is every pair (j, k) of i's own list
// with d_jk < R_j + R_k.  So the wavefront puts its list's atoms and weights in LDS once
// and computes the pairs from there: lane (k mod 16, j mod 4) holds up to three k and
// walks the j, recomputing the overlap s_jk (one reciprocal square root) instead of
// fetching it; sums over j alone (the k's share of the derivative) and over k alone
// (SASA_i's own terms) stay in registers.  It is bound by FP64 issue (38 instructions a
// pair; four wavefronts a SIMD, 128 registers).  Gathering each j's list and overlaps
// from memory instead waited on loads most of its time: average over the steps of a run
// (a full update every fifth) on 256 chains 241 -> 116 us, 64 replicas 69 -> 39; a full
// update of a 300-residue chain 46 -> 24, of a 20-residue chain 26 -> 12.
//
// EONLY (calcLCPOSasaEnergies, lcpo.cpp:522-556: the SASA alone, with k excluded
// when (R_i + R_k) < d_ik) and atoms with a cut list take the pairs from the
// neighbours' lists: lanes take (j, k) pairs in turn after a first pass over j has put
// the weights in LDS.  All sums are reduced over the wave in a fixed order.
constexpr int kLcpoDepth = 4;  // (j, k) tasks per lane in flight when gathering
// waves of k_lcpo_sasa (each walks atoms blockIdx.x, + gridDim.x, ...)
constexpr int kLcpoGrid = 65536;

// 1 / sqrt(x) in FP64: the hardware's estimate y (relative error 2^-24) with one step of
// third order, y (1 + e/2 + 3 e^2/8) with e = 1 - x y^2 (what is left: e^3, below 2^-70)
__device__ __forceinline__ double rsqrt_fp64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y, e * fma(0.375, e, 0.5), y);
}

// A neighbour of i in LDS, as seven 16-byte arrays (consecutive j: no bank conflicts)
struct LcpoLds {
  double2 xy[kLcpoMax], zr[kLcpoMax];      // position, R
  double2 w34[kLcpoMax], sw[kLcpoMax];     // P3 sigma, P4 sigma | s_ij, P4 sigma s_ji
  double2 dxy[kLcpoMax], dza[kLcpoMax];    // d s_ji / d x_i (its j part): x, y | z, x of the i part
  double2 ayz[kLcpoMax];                   // the i part (d s_ij / d x_i): y, z
};

// The pairs (j, k) of the list with k = 16 m + (lane & 15), m0 <= m < m0 + MB.
template <int MB>
__device__ __forceinline__ void lcpo_pairs(const LcpoLds &L, int n, int m0, int lane, double der[3], double a4[3],
                                           double &Si3, double &Si4) {
  const double PI = Consts::PI;
  double xk[MB], yk[MB], zk[MB], rk[MB], hk[MB];
  double c3[MB], ca[MB], cb[MB], vx[MB], vy[MB], vz[MB];
  int kk[MB];
#pragma unroll
  for (int m = 0; m < MB; m++) {
    const int k = 16 * (m0 + m) + (lane & 15);
    kk[m] = min(k, n - 1);
    const double2 a = L.xy[kk[m]], b = L.zr[kk[m]];
    xk[m] = k < n ? a.x : 1e30;  // a pad overlaps nothing
    yk[m] = a.y;
    zk[m] = b.x;
    rk[m] = b.y;
    hk[m] = 0.5 * b.y * b.y;
    c3[m] = ca[m] = cb[m] = vx[m] = vy[m] = vz[m] = 0.0;
  }
  for (int j0 = 0; j0 < n; j0 += 4) {
    const int j = min(j0 + (lane >> 4), n - 1);
    const double2 a = L.xy[j], b = L.zr[j], w = L.w34[j], s2 = L.sw[j], d01 = L.dxy[j], d2a = L.dza[j], a12 = L.ayz[j];
    const double xj = j0 + (lane >> 4) < n ? a.x : -1e30;
    const double rj = b.y, hj = 0.5 * rj * rj, cj = 2.0 * PI * rj;
    double T = 0.0;
#pragma unroll
    for (int m = 0; m < MB; m++) {
      double d2, lim;
      {
#pragma clang fp contract(off)
        const double g = xj - xk[m], h = a.y - yk[m], q = b.x - zk[m];
        d2 = g * g + h * h + q * q;  // the list's test, bit for bit
        lim = (rj + rk[m]) * (rj + rk[m]);
      }
      const bool on = d2 < lim && kk[m] != j;
      const double inv = rsqrt_fp64(d2);
      const double d = d2 * inv;
      const double s0 = cj * fma(-(hj - hk[m]), inv, fma(-0.5, d, rj));
      const double s = on ? s0 : 0.0, o = on ? 1.0 : 0.0;
      T += s;
      c3[m] = fma(o, w.x, c3[m]);
      ca[m] = fma(o, s2.y, ca[m]);
      cb[m] = fma(w.y, s, cb[m]);
      const double ow = o * w.y;
      vx[m] = fma(ow, d01.x, vx[m]);
      vy[m] = fma(ow, d01.y, vy[m]);
      vz[m] = fma(ow, d2a.x, vz[m]);
    }
    Si3 += T;
    Si4 = fma(s2.x, T, Si4);
    a4[0] = fma(T, d2a.y, a4[0]);
    a4[1] = fma(T, a12.x, a4[1]);
    a4[2] = fma(T, a12.y, a4[2]);
  }
#pragma unroll
  for (int m = 0; m < MB; m++) {
    const int k = kk[m];
    if (16 * (m0 + m) + (lane & 15) >= n) continue;
    // s_ik, its derivatives with respect to x_i (i part, k part)
    const double s = L.sw[k].x, p1 = c3[m] + ca[m], p2 = c3[m] + cb[m];
    const double2 d01 = L.dxy[k], d2a = L.dza[k], a12 = L.ayz[k];
    der[0] += fma(p1, d2a.y, fma(p2, d01.x, s * vx[m]));
    der[1] += fma(p1, a12.x, fma(p2, d01.y, s * vy[m]));
    der[2] += fma(p1, a12.y, fma(p2, d2a.x, s * vz[m]));
  }
}

template <bool EONLY>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_lcpo_sasa(int n, const double4 *__restrict__ pr, const int8_t *__restrict__ use,
                                                  const double4 *__restrict__ P,
                                                  const double *__restrict__ sig, const int *__restrict__ nl_cnt,
                                                  const int *__restrict__ nl_idx, const double *__restrict__ nl_s,
                                                  double *__restrict__ sasa, double *__restrict__ dvx,
                                                  double *__restrict__ dvy, double *__restrict__ dvz) {
#pragma clang fp contract(off)
  // gathering: jw holds s_ji, P3 sigma, P4 sigma, Si2_t, d2(3), a2t(3) of each j
  __shared__ __align__(16) union {
    LcpoLds list;
    struct {
      int jidx[kLcpoMax], joff[kLcpoMax + 1];
      double jw[kLcpoMax][10];
    } g;
  } sh;
  auto &jidx = sh.g.jidx;
  auto &joff = sh.g.joff;
  auto &jw = sh.g.jw;
  const int lane = threadIdx.x;
  // at most kLcpoGrid waves walk the atoms; on the steps that re-apply stored
  // forces every wave returns at the test above
  for (int i = blockIdx.x; i < n; i += gridDim.x) {
  __syncthreads();  // the LDS tables of the previous atom are no longer read
  if (!use[i]) {
    if (lane == 0) {
      sasa[i] = 0.0;
      if (!EONLY) dvx[i] = dvy[i] = dvz[i] = 0.0;
    }
    continue;
  }
  const double PI = Consts::PI, TwoPI = 2.0 * Consts::PI, FourPI = 4.0 * Consts::PI;
  const double4 pi4 = pr[i];
  const double pix = pi4.x, piy = pi4.y, piz = pi4.z;
  const double ri = pi4.w;
  const int ni = nl_cnt[i] & (kListCut - 1);
  double der[3] = {0, 0, 0}, a2[3] = {0, 0, 0}, a4[3] = {0, 0, 0};
  double Si2 = 0, Si3 = 0, Si4 = 0;
  // whole lists (uniform over the wave)?
  bool gather = EONLY;
  if (!EONLY) {
    int cut = nl_cnt[i] & kListCut;
    for (int jn = lane; jn < ni; jn += 64) cut |= nl_cnt[nl_idx[(size_t)i * kLcpoMax + jn]] & kListCut;
    gather = __ballot(cut != 0) != 0ull;
  }
  // pass over j: per-j weights, and the k counts when gathering
  for (int jn = lane; jn < ni; jn += 64) {
    const int ja = nl_idx[(size_t)i * kLcpoMax + jn];
    double Si2_t = 0.0;
    if (EONLY) {
      Si2_t = nl_s[(size_t)i * kLcpoMax + jn];
      Si2 += Si2_t;
      jw[jn][3] = Si2_t;
    }
    if (gather) {
      jidx[jn] = ja;
      joff[jn + 1] = nl_cnt[ja] & (kListCut - 1);
    }
    if (!EONLY) {
      const double4 pj4 = pr[ja];
      const double pjx = pj4.x, pjy = pj4.y, pjz = pj4.z;
      const double gx = pjx - pix, gy = pjy - piy, gz = pjz - piz;
      const double dij = sqrt(gx * gx + gy * gy + gz * gz);
      const double rj = pj4.w;
      const double inv = 1 / dij;
      double t = 0.5 * (ri * ri - rj * rj) * inv;
      Si2_t = TwoPI * ri * (ri - dij * 0.5 - t);
      Si2 += Si2_t;
      const double sji = TwoPI * rj * (rj - dij * 0.5 + t);
      t *= 2.0 * inv;
      const double ddd[3] = {-(pix - pjx) / dij, -(piy - pjy) / dij, -(piz - pjz) / dij};
      const double dAj = PI * rj * (-t - 1), dAi = PI * ri * (t - 1);
      const double4 Pj = P[ja];
      const double sj = sig[ja];
      double d2[3], a2t[3];
      for (int c = 0; c < 3; c++) {
        d2[c] = dAj * ddd[c];
        a2t[c] = dAi * ddd[c];
        der[c] += d2[c] * (Pj.y * sj);  // the P2 term of SASA_j
        a2[c] += a2t[c];
      }
      if (gather) {
        jw[jn][0] = sji;
        jw[jn][1] = Pj.z * sj;
        jw[jn][2] = Pj.w * sj;
        jw[jn][3] = Si2_t;
        for (int c = 0; c < 3; c++) {
          jw[jn][4 + c] = d2[c];
          jw[jn][7 + c] = a2t[c];
        }
      } else {
        sh.list.xy[jn] = make_double2(pjx, pjy);
        sh.list.zr[jn] = make_double2(pjz, rj);
        sh.list.w34[jn] = make_double2(Pj.z * sj, Pj.w * sj);
        sh.list.sw[jn] = make_double2(Si2_t, Pj.w * sj * sji);
        sh.list.dxy[jn] = make_double2(d2[0], d2[1]);
        sh.list.dza[jn] = make_double2(d2[2], a2t[0]);
        sh.list.ayz[jn] = make_double2(a2t[1], a2t[2]);
      }
    }
  }
  __syncthreads();
  if (!gather) {
    for (int m0 = 0; 16 * m0 < ni; m0 += 3) {
      const int left = (ni + 15) / 16 - m0;
      if (left >= 3)
        lcpo_pairs<3>(sh.list, ni, m0, lane, der, a4, Si3, Si4);
      else if (left == 2)
        lcpo_pairs<2>(sh.list, ni, m0, lane, der, a4, Si3, Si4);
      else
        lcpo_pairs<1>(sh.list, ni, m0, lane, der, a4, Si3, Si4);
    }
  } else {
  if (lane == 0) {  // exclusive prefix of the k counts, in j order
    joff[0] = 0;
    for (int jn = 0; jn < ni; jn++) joff[jn + 1] += joff[jn];
  }
  __syncthreads();
  const int total = joff[ni];
  // the (j, k) tasks, kLcpoDepth per lane at a time with every load of the
  // batch issued before the arithmetic (the gathers, not the arithmetic, set the pace)
  int jn = 0;
  for (int t0 = lane; t0 < total; t0 += 64 * kLcpoDepth) {
    int jnv[kLcpoDepth], kav[kLcpoDepth];
    double sjkv[kLcpoDepth];
#pragma unroll
    for (int u = 0; u < kLcpoDepth; u++) {
      const int t = t0 + 64 * u;
      kav[u] = i;  // no task
      jnv[u] = 0;
      sjkv[u] = 0.0;
      if (t < total) {
        while (joff[jn + 1] <= t) jn++;  // t only grows, so j only moves forward
        const int ja = jidx[jn];
        const int kn = t - joff[jn];
        jnv[u] = jn;
        kav[u] = nl_idx[(size_t)ja * kLcpoMax + kn];
        if (EONLY) sjkv[u] = nl_s[(size_t)ja * kLcpoMax + kn];
      }
    }
    double4 pkv[kLcpoDepth];
#pragma unroll
    for (int u = 0; u < kLcpoDepth; u++) pkv[u] = pr[kav[u]];
#pragma unroll
    for (int u = 0; u < kLcpoDepth; u++) {
    const int ka = kav[u];
    if (ka == i) continue;
    const int jn_u = jnv[u];
    const double4 pk4 = pkv[u];
    const double pkx = pk4.x, pky = pk4.y, pkz = pk4.z;
    const double rk = pk4.w;
    const double hx = pkx - pix, hy = pky - piy, hz = pkz - piz;
    double dik = hx * hx + hy * hy + hz * hz;
    double sjk = sjkv[u];
    if (!EONLY) {  // the overlap of j with k, as the neighbour's list would hold it
      const double4 pj4 = pr[jidx[jn_u]];
      const double gx = pj4.x - pkx, gy = pj4.y - pky, gz = pj4.z - pkz;
      const double d = sqrt(gx * gx + gy * gy + gz * gz);
      sjk = TwoPI * pj4.w * (pj4.w - d * 0.5 - 0.5 * (pj4.w * pj4.w - rk * rk) * (1 / d));
    }
    if (EONLY) {
      if ((ri + rk) < sqrt(dik)) continue;
    } else {
      if ((ri + rk) * (ri + rk) < dik) continue;
    }
    Si3 += sjk;
    Si4 += jw[jn_u][3] * sjk;
    if (EONLY) continue;
    dik = sqrt(dik);
    const double invik = 1 / dik;
    const double uu = (ri * ri - rk * rk) * (invik * invik);
    const double dA1 = PI * ri * (uu - 1);
    const double dA2 = PI * rk * (-uu - 1);
    const double s3ik = PI * ri * (2 * ri - dik - dik * uu);
    const double dk[3] = {-(pix - pkx) * invik, -(piy - pky) * invik, -(piz - pkz) * invik};
    const double c3 = jw[jn_u][1], c4 = jw[jn_u][2], sji = jw[jn_u][0];
    for (int c = 0; c < 3; c++) {
      der[c] += c3 * (dA1 * dk[c] + dA2 * dk[c]);                          // P3 term of SASA_j
      der[c] += c4 * (sji * (dA1 * dk[c]) + sjk * dA2 * dk[c] + jw[jn_u][4 + c] * s3ik);  // P4 term of SASA_j
      a4[c] += sjk * jw[jn_u][7 + c];
    }
    }
  }
  }
  // SASA and derivative are linear in the sums: combined per lane, then added over the wave
  const double4 Pi = P[i];
  const double Si = FourPI * ri * ri;
  double SAi = Pi.x * Si + wave_sum(Pi.y * Si2 + Pi.z * Si3 + Pi.w * Si4);
  if (!EONLY) {
    const double k2 = Pi.y * sig[i], k4 = Pi.w * sig[i];
    for (int c = 0; c < 3; c++) der[c] = wave_sum(der[c] + a2[c] * k2 + a4[c] * k4);
  }
  if (lane != 0) continue;
  if (SAi < 0) {  // LCPO can go negative for buried atoms (lcpo.cpp:940-944)
    SAi = 0;
    der[0] = der[1] = der[2] = 0.0;
  }
  sasa[i] = SAi;
  if (EONLY) continue;  // the stored derivatives of the last force evaluation stay
  dvx[i] = der[0];
  dvy[i] = der[1];
  dvz[i] = der[2];
  }
}

// The block's sum of v in a tree (256 threads, s: 256 doubles), as its 4-wide partial.
__device__ __forceinline__ void block_sum_256(double v, double *s, double *part) {
  s[threadIdx.x] = v;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 4) part[4 * blockIdx.x + threadIdx.x] = threadIdx.x == 0 ? s[0] : 0.0;
}

// Adds the stored derivatives (J/A per molecule) as forces in fixed point
// (kcal/mol/A) and writes each atom's sigma * SASA in kcal/mol.
// With `part` also each block's energy sum (4-wide, the first slot used), and after the
// atoms' blocks two that take a GB evaluation's energy sums: three launches in one.
__global__ __launch_bounds__(256) void k_lcpo_apply(int n, double to_kcal, const double *__restrict__ sasa, const double *__restrict__ sig,
                             const double *__restrict__ dvx, const double *__restrict__ dvy,
                             const double *__restrict__ dvz, long long *__restrict__ fx, long long *__restrict__ fy,
                             long long *__restrict__ fz, double *__restrict__ eatom, double *__restrict__ part,
                             GBSums G) {
  __shared__ double s[4][256];
  const int blocks = (n + 255) / 256;
  if ((int)blockIdx.x >= blocks) {
    gb_sums_block(G, 0, (int)blockIdx.x - blocks, s);
    return;
  }
  const int i = blockIdx.x * 256 + threadIdx.x;
  double e = 0.0;
  if (i < n) {
    e = sasa[i] * sig[i] * to_kcal;
    eatom[i] = e;
    const double gx = dvx[i], gy = dvy[i], gz = dvz[i];
    if (gx != 0.0 || gy != 0.0 || gz != 0.0) {
      // to the nearest unit (fix_from_double rounds down): surface forces are small
      const double half = 0.5 / kFixScale;
      fix_add(&fx[i], fix_from_double(fma(gx, to_kcal, half)));
      fix_add(&fy[i], fix_from_double(fma(gy, to_kcal, half)));
      fix_add(&fz[i], fix_from_double(fma(gz, to_kcal, half)));
    }
  }
  if (part) block_sum_256(e, s[0], part);
}

__global__ void k_lcpo_energy(int n, double to_kcal, const double *__restrict__ sasa, const double *__restrict__ sig,
                              double *__restrict__ eatom) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) eatom[i] = sasa[i] * sig[i] * to_kcal;
}

}  // namespace

void LCPOState::add_system(int first, int count, const int8_t *use, const double *radius, const double *P4,
                           const double *sigma_j) {
  for (int a = 0; a < count; a++) {
    h_use.push_back(use[a] ? 1 : 0);
    h_R.push_back(radius[a] + 1.4);  // FF_SASA_LCPO::setup, lcpo.cpp:107
    for (int c = 0; c < 4; c++) h_P.push_back(P4[4 * a + c]);
    h_sig.push_back(sigma_j[a]);
    h_atom_sys.push_back((int)h_first.size());
  }
  h_first.push_back(first);
  h_count.push_back(count);
  n = (int)h_use.size();
}

void LCPOState::append(const LCPOState &o, int first) {
  const int sys = (int)h_first.size();
  h_use.insert(h_use.end(), o.h_use.begin(), o.h_use.end());
  h_R.insert(h_R.end(), o.h_R.begin(), o.h_R.end());
  h_P.insert(h_P.end(), o.h_P.begin(), o.h_P.end());
  h_sig.insert(h_sig.end(), o.h_sig.begin(), o.h_sig.end());
  h_atom_sys.insert(h_atom_sys.end(), o.n, sys);
  h_first.push_back(first);
  h_count.push_back(o.n);
  n = (int)h_use.size();
}

void LCPOState::upload(hipStream_t s) {
  max_R = 0.0;
  for (int a = 0; a < n; a++)
    if (h_use[a]) max_R = std::max(max_R, h_R[a]);
  use.upload(h_use, s);
  R.upload(h_R, s);
  std::vector<double4> p4(n);
  for (int a = 0; a < n; a++) p4[a] = make_double4(h_P[4 * a], h_P[4 * a + 1], h_P[4 * a + 2], h_P[4 * a + 3]);
  P.upload(p4, s);
  sig.upload(h_sig, s);
  atom_sys.upload(h_atom_sys, s);
  sys_first.upload(h_first, s);
  sys_count.upload(h_count, s);
  pr.resize(n);  // allocated here: run() may be recorded into a graph
  tile_box.resize((size_t)6 * ((n + 63) / 64));
  nl_cnt.resize(n);
  nl_idx.resize((size_t)n * kLcpoMax);
  nl_s.resize((size_t)n * kLcpoMax);
  sasa.resize(n);
  dvx.resize(n);
  dvy.resize(n);
  dvz.resize(n);
  eatom.resize(n);
  std::vector<double> zero(n, 0.0);  // nothing to re-apply before the first full step
  sasa.upload(zero, s);
  dvx.upload(zero, s);
  dvy.upload(zero, s);
  dvz.upload(zero, s);
}

void LCPOState::run(hipStream_t s, const double *x, const double *y, const double *z, long long *fx, long long *fy,
                    long long *fz, int step, bool full, bool energy_only, double *block_part, const GBSums *gb) {
  auto apply = [&]() {
    hipLaunchKernelGGL(k_lcpo_apply, dim3((n + 255) / 256 + (gb ? 2 : 0)), dim3(256), 0, s, n,
                       Consts::J_to_kcalmol(), sasa.p, sig.p, dvx.p, dvy.p, dvz.p, fx, fy, fz, eatom.p, block_part,
                       gb ? *gb : GBSums{});
    PDGPU_HIP(hipGetLastError());
  };
  if (!full && !energy_only && reapplies(step)) {  // the stored forces again
    apply();
    return;
  }
  hipLaunchKernelGGL(k_lcpo_pack, dim3((n + 255) / 256), dim3(256), 0, s, n, x, y, z, use.p, R.p,
                     pr.p, tile_box.p);
  const int lb = std::min((n + kListWaves - 1) / kListWaves, kListGrid);
  if (energy_only) {
    hipLaunchKernelGGL(k_lcpo_lists<true>, dim3(lb), dim3(64 * kListWaves), 0, s, n, atom_sys.p, sys_first.p,
                       sys_count.p, pr.p, tile_box.p, max_R, nl_cnt.p, nl_idx.p, nl_s.p);
    hipLaunchKernelGGL(k_lcpo_sasa<true>, dim3(std::min(n, kLcpoGrid)), dim3(64), 0, s, n, pr.p, use.p, P.p, sig.p,
                       nl_cnt.p, nl_idx.p, nl_s.p, sasa.p, dvx.p, dvy.p, dvz.p);
    hipLaunchKernelGGL(k_lcpo_energy, dim3((n + 255) / 256), dim3(256), 0, s, n, Consts::J_to_kcalmol(), sasa.p,
                       sig.p, eatom.p);
  } else {
    hipLaunchKernelGGL(k_lcpo_lists<false>, dim3(lb), dim3(64 * kListWaves), 0, s, n, atom_sys.p, sys_first.p,
                       sys_count.p, pr.p, tile_box.p, max_R, nl_cnt.p, nl_idx.p, nl_s.p);
    hipLaunchKernelGGL(k_lcpo_sasa<false>, dim3(std::min(n, kLcpoGrid)), dim3(64), 0, s, n, pr.p, use.p, P.p, sig.p,
                       nl_cnt.p, nl_idx.p, nl_s.p, sasa.p, dvx.p, dvy.p, dvz.p);
    apply();
  }
  PDGPU_HIP(hipGetLastError());
}

}  // namespace pdgpu

namespace pdgpu {

namespace {
// Sums per-atom energies into per-block partials (4 per block, first slot used).
__global__ void k_block_sum(int n, const double *__restrict__ v, double *__restrict__ part) {
  __shared__ double s[256];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  block_sum_256(i < n ? v[i] : 0.0, s, part);
}
}  // namespace

void Engine::launch_lcpo(double *energy_slot, int step, bool full, bool energy_only, const GBSums *with_gb) {
  require(lcpo != nullptr, "LCPO component not set up");
  // lcpo.cpp takes every distance as p_j - p_i with no image
  require(!periodic, "LCPO runs in vacuum: PD's LCPO takes raw displacements, no periodic images");
  const int blocks = (n + 255) / 256;
  e_partial_lcpo.resize((size_t)blocks * 4);
  {
    ScopedTimer t(*this, "lcpo");
    lcpo->run(stream, x.p, y.p, z.p, fbx.p, fby.p, fbz.p, step, full, energy_only, e_partial_lcpo.p,
              with_gb);
  }
  if (energy_only) hipLaunchKernelGGL(k_block_sum, dim3(blocks), dim3(256), 0, stream, n, lcpo->eatom.p, e_partial_lcpo.p);
  defer_sum4(e_partial_lcpo.p, blocks, energy_slot);
}

}  // namespace pdgpu

using pdgpu::Engine;

extern "C" int pdgpu_setup_lcpo(pdgpu_engine *h, const pdgpu_lcpo_params *p, const double *radius, const double *P,
                                const int8_t *use, const double *asp) {
  Engine *E = reinterpret_cast<Engine *>(h);
  if (!E) return PDGPU_ERR_ARG;
  if (!p || !radius || !P || !use) {
    E->last_error = "pdgpu_setup_lcpo: null argument";
    return PDGPU_ERR_ARG;
  }
  try {
    PDGPU_HIP(hipSetDevice(E->device));
    auto L = std::make_unique<pdgpu::LCPOState>();
    L->update = p->UpdateSasa;
    // sigma = ASP / Na / J2kcal: J per A^2 per molecule (lcpo.cpp:63)
    std::vector<double> sig(E->n);
    for (int a = 0; a < E->n; a++)
      sig[a] = (asp ? asp[a] : p->GlobalASP) / pdgpu::Consts::Na / pdgpu::Consts::J2kcal();
    L->add_system(0, E->n, use, radius, P, sig.data());
    L->upload(E->stream);
    E->sync();
    E->lcpo = std::move(L);
    return PDGPU_OK;
  } catch (const pdgpu::EngineError &x) {
    E->last_error = x.what();
    return x.code;
  } catch (const std::exception &x) {
    E->last_error = x.what();
    return PDGPU_ERR_SETUP;
  }
}

extern "C" int pdgpu_get_sasa(pdgpu_engine *h, double *sasa) {
  Engine *E = reinterpret_cast<Engine *>(h);
  if (!E || !sasa) return PDGPU_ERR_ARG;
  if (!E->lcpo) {
    E->last_error = "LCPO component not set up";
    return PDGPU_ERR_ARG;
  }
  try {
    E->lcpo->sasa.download(sasa, E->n, E->stream);
    E->sync();
    return PDGPU_OK;
  } catch (const pdgpu::EngineError &x) {
    E->last_error = x.what();
    return x.code;
  }
}
