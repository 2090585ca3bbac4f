// k_gb.hip -- FF_GeneralizedBorn_Still on the device, for one system or a batch
// of independent systems.
//
// PD evaluates three passes over its (shadow) neighbour list each step:
//   1. calcBornRadii_PairwiseApprox (gbff.cpp:432-483): Gpol_i = terms123_i +
//      sum_j P4 Vj CCF / r^4 over non-bonded/1-4 partners within GbsaStillCutoff,
//      a_i = -halfeconv / Gpol_i + BornRadiusOffset;
//   2. the pair pass of calcForcesIncludingVacuo (gbff.cpp:1546-1746): the Still
//      cross term premul q_i q_j / sqrt(r^2 + a_i a_j exp(-r^2/4 a_i a_j)) with its
//      dE/dr and dE/d(a_i a_j), vacuum Coulomb (eps_solvent where the GB term is
//      dropped, uGB <= ExpApproxThreshold), LJ, energy switching, plus the self
//      terms premul q^2 / a (gbff.cpp:1750-1757);
//   3. the Born-radius chain rule (gbff.cpp:1768-1825) with gpi = a_i^2 / 166.0.
// Here every pass is an all-pairs walk over 64x64 atom tiles of each system
// (upper triangle of tile pairs): lanes hold the i atoms, the j tile sits in LDS
// and is visited in the rotated order j = (lane + t) mod 64.
//
// What bounds the passes is VALU issue (a wave64 instruction holds its SIMD for
// four cycles), so a tile pair runs the shortest loop its geometry allows.  One
// small kernel per evaluation gives every tile a centre and a radius; from these
// (and the tiles' largest GB and Born radii) a tile pair is
//   far   every pair lies inside all cutoffs and beyond the reach of the short-range
//         part of the pass (the exp threshold of the cross term, the CCF function of
//         the radii): no tests, and only the terms that are left (the pair pass:
//         solvent Coulomb and LJ).  Two i tiles share each j read.  FP32
//         displacements from FP32 offsets about the midpoint of the two tiles,
//         which the distance of the tiles keeps at the precision of r itself;
//   near  everything else: FP64 displacements and r^2, rounded once, with PD's per-pair
//         cutoff tests unless every pair is inside them;
//   out   beyond every cutoff: left at once.
// Tile pairs whose atoms lie within BondOrder::m_MaxIndexDelta of each other, or
// hold an off-diagonal covalent partner, and the diagonal ones are tasks of their
// own with a table of 2-bit codes (in the rotated order, built once at setup), so
// the loop looks no bond order up.
// The j partial sums stay in registers and move with the rotation: acc =
// rotate(acc) + term is one DPP add.  Every 16 steps (a chunk) the FP32 partial
// sums go to 64-bit fixed point; chunks, tasks and wavefronts then only add
// integers, so forces, radii and dE/da are the same bits for every work split.
// Measured (radii / pair / chain): 256 chains of 20-120 residues (54,560 tile pairs) 243
// / 467 / 299 -> 101 / 304 / 170 us, both sums of the pair pass at 0.95 of the VALU issue
// rate; a 300-residue chain 36 / 55 / 44 -> 14 / 31 / 22 us; a 20-residue chain at 15 A
// cutoffs 34 / 45 / 36 -> 9 / 16 / 11 us, where the latency of one wavefront's 16 steps is
// what is left.  The near loops' 1 / r^2 to full FP32 precision and the FP64 decision at the
// exp threshold cost 30 of the 304 us; they take the forces' error against FP64 from 5.6e-7 to
// 3.5e-7 (20 residues) and 1.1e-6 to 3.8e-7 (300 residues).
#include <algorithm>
#include <array>
#include <cmath>
#include <map>
#include <mutex>
#include <tuple>

#include "bonded_dev.hpp"
#include "engine.hpp"

namespace pdgpu {

namespace {

constexpr int kTile = 64;
constexpr int kChunk = 16;  // rotated steps between two conversions to fixed point
// codes of a pair in a task's table: 0 non-bonded, 1 1-4 partner, 2 1-2 or 1-3
// partner, 3 no pair (beyond the tile's atoms, or a diagonal pair taken elsewhere)
enum { kPairPlain = 0, kPair14 = 1, kPairBonded = 2, kPairNone = 3 };

// Bond order of pair (a, b) as NeighbourList::calcNewList + correctOffDiagonalBondOrders
// assign it (neighbourlist.cpp:399-406, 179-220); indices are local to the system.
__device__ __forceinline__ int gb_bond_order(int a, int b, int mid, const int8_t *__restrict__ band,
                                             const int *__restrict__ sp_off, const int *__restrict__ sp_part,
                                             const int *__restrict__ sp_ord) {
  int hi = max(a, b), lo = min(a, b);
  int bo = 7;
  if (hi - lo < mid) bo = band[(long)lo * mid + (hi - lo - 1)];
  for (int k = sp_off[lo]; k < sp_off[lo + 1]; k++)
    if (sp_part[k] == hi) bo = sp_ord[k];
  return bo & 7;
}

// The code tables of the tasks with codes (once, at setup): one wavefront per
// task, word c * 64 + lane holds lane's codes of steps 16 c .. 16 c + 15.
__global__ __launch_bounds__(64) void k_gb_codes(const GBTask *__restrict__ tasks, const int *__restrict__ coded,
                                                 const int2 *__restrict__ tile_atoms, const GBSys *__restrict__ sys,
                                                 const int8_t *__restrict__ band, const int *__restrict__ sp_off,
                                                 const int *__restrict__ sp_part, const int *__restrict__ sp_ord,
                                                 unsigned *__restrict__ codes) {
  const GBTask w = tasks[coded[blockIdx.x]];
  const GBSys S = sys[w.sys];
  const int2 A = tile_atoms[w.ti], B = tile_atoms[w.tj];
  const bool diag = w.ti == w.tj;
  const int lane = threadIdx.x;
  for (int c = 0; c < kTile / kChunk; c++) {
    unsigned word = 0u;
    for (int u = 0; u < kChunk; u++) {
      const int t = c * kChunk + u, jj = (lane + t) & (kTile - 1);
      bool v = lane < A.y && jj < B.y;
      if (diag) v = v && ((t >= 1 && t < 32) || (t == 32 && lane < 32));
      unsigned code = kPairNone;
      if (v) {
        const int bo = gb_bond_order(A.x + lane - S.first, B.x + jj - S.first, S.mid, band + S.band_off,
                                     sp_off + S.sp_base, sp_part, sp_ord);
        code = bo <= 2 ? kPairBonded : (bo == 3 ? kPair14 : kPairPlain);
      }
      word |= code << (2 * u);
    }
    codes[(size_t)w.code * (kTile / kChunk) * kTile + c * kTile + lane] = word;
  }
}

// Opens an evaluation: each tile's centre (of its atoms' box) and the largest
// distance of an atom from it, its largest GB radius; clears the Gpol sums.  One
// wavefront per tile.
//
// The launch opens an evaluation: its first workgroups take the bonded terms (FP64 chains
// of a few us that no other kernel depends on), its last the previous MD step's energy
// sums.  With those launches gone, and the GB and surface energy sums in the launch of
// the surface forces, a step of a 20-residue chain takes 64 us where it took 85.
__global__ __launch_bounds__(256) void k_gb_open(int ntiles, const int2 *__restrict__ tile_atoms,
                                                 const double *__restrict__ x, const double *__restrict__ y,
                                                 const double *__restrict__ z, const float *__restrict__ gbrad,
                                                 GBTile *__restrict__ tiles, long long *__restrict__ gpol,
                                                 BondedArrays B, int bonded, long long *__restrict__ fx,
                                                 long long *__restrict__ fy, long long *__restrict__ fz,
                                                 double *__restrict__ bonded_partial,
                                                 double *__restrict__ bonded_eterm, SumList L) {
  __shared__ long long window[3 * kBondedWindow];
  if ((int)blockIdx.x < bonded) {
    bonded_block((int)blockIdx.x, B, x, y, z, fx, fy, fz, bonded_partial, bonded_eterm, window);
    return;
  }
  if ((L.n > 0 || L.record) && blockIdx.x == gridDim.x - 1) {
    sum_lists<true>(L);
    return;
  }
  const int t = ((int)blockIdx.x - bonded) * 4 + ((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= ntiles) return;  // whole waves; no barrier follows
  const int2 A = tile_atoms[t];
  const bool on = lane < A.y;
  const int i = A.x + lane;
  double p[3] = {0.0, 0.0, 0.0}, c[3];
  float R = 0.0f;
  if (on) {
    p[0] = x[i];
    p[1] = y[i];
    p[2] = z[i];
    R = gbrad[i];
    gpol[i] = 0;
  }
  double d2 = 0.0;
  for (int k = 0; k < 3; k++) {
    c[k] = 0.5 * (wave_min(on ? p[k] : 1e300) + wave_max(on ? p[k] : -1e300));
    d2 += (p[k] - c[k]) * (p[k] - c[k]);
  }
  const double rad = wave_max(on ? sqrt(d2) : 0.0);
  const double rmax = wave_max((double)R);
  if (lane == 0) {
    GBTile T;
    T.x = c[0];
    T.y = c[1];
    T.z = c[2];
    T.rad = rad;
    T.rmax = (float)rmax;
    T.amax = 0.0f;
    tiles[t] = T;
  }
}

// a_i = -halfeconv / (terms123_i + sum) + BornRadiusOffset; the self term
// premul q^2 / a seeds dE/da (gbff.cpp:1750-1757).  One wavefront per tile: also the
// tile's largest Born radius (infinite, so that no tile pair counts as far, when one is
// not positive).
__global__ __launch_bounds__(256) void k_gb_finalize_radii(int ntiles, const int2 *__restrict__ tile_atoms,
                                                           double halfeconv, double offset, double premul,
                                                           const double *__restrict__ terms123,
                                                           const long long *__restrict__ gpol,
                                                           const float *__restrict__ q, double *__restrict__ born,
                                                           float *__restrict__ bornf, long long *__restrict__ deda,
                                                           double *__restrict__ eself, GBTile *__restrict__ tiles) {
  const int t = blockIdx.x * 4 + ((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= ntiles) return;  // whole waves; no barrier follows
  const int2 A = tile_atoms[t];
  const int i = A.x + lane;
  double amax = 0.0;
  if (lane < A.y) {
    const double G = terms123[i] + (double)gpol[i] * (1.0 / kFixScale);
    const double a = -halfeconv / G + offset;
    born[i] = a;
    bornf[i] = (float)a;
    const double qi = q[i];
    const double epol = premul * qi * qi / a;
    eself[i] = epol;
    deda[i] = fix_from_double(-epol / a);
    amax = a > 0.0 ? a : 1e30;
  }
  amax = wave_max(amax);
  if (lane == 0) tiles[t].amax = (float)amax;
}

// The value of the next lane (lane 63 takes lane 0's): what the rotation of the j
// atoms by one step asks of their partial sums.  Feeding an add, it costs nothing.
__device__ __forceinline__ float rotate1(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x134 /* wave_rol:1 */, 0xf, 0xf, true));
}

// sin and cos of h in [0, pi/2]: Taylor polynomials to h^13 and h^14 (remainder below 1e-9)
__device__ __forceinline__ float sin_quarter(float h) {
  const float s = h * h;
  float p = fmaf(s, 1.0f / 6227020800.0f, -1.0f / 39916800.0f);
  p = fmaf(s, p, 1.0f / 362880.0f);
  p = fmaf(s, p, -1.0f / 5040.0f);
  p = fmaf(s, p, 1.0f / 120.0f);
  p = fmaf(s, p, -1.0f / 6.0f);
  return fmaf(h * s, p, h);
}
__device__ __forceinline__ float cos_quarter(float h) {
  const float s = h * h;
  float p = fmaf(s, -1.0f / 87178291200.0f, 1.0f / 479001600.0f);
  p = fmaf(s, p, -1.0f / 3628800.0f);
  p = fmaf(s, p, 1.0f / 40320.0f);
  p = fmaf(s, p, -1.0f / 720.0f);
  p = fmaf(s, p, 1.0f / 24.0f);
  p = fmaf(s, p, -0.5f);
  return fmaf(s, p, 1.0f);
}

// gpi dE/da_i P4 with gpi = a_i^2 / 166.0 (gbff.cpp:1772), dE/da from its fixed-point sum
__device__ __forceinline__ float chain_weight(const double *__restrict__ born, const long long *__restrict__ deda,
                                              int i, float P4) {
  const double a = born[i];
  const double gpi = -(a * a) / -166.0;
  return (float)(gpi * ((double)deda[i] * (1.0 / kFixScale)) * (double)P4);
}

// max(a, |b|), NaN if b is
__device__ __forceinline__ float fmax_nan(float a, float b) { return fabsf(b) <= a ? a : fabsf(b); }

// 1 / r^2 to FP32 rounding: r2f the rounded r^2, r2lo what the rounding took.  The LJ
// terms raise it to the 6th and 7th power; taken from the hardware's reciprocal square
// root (1 ulp, biased) its error was the largest part of the forces' error.
__device__ __forceinline__ float rcp_near(float r2f, float r2lo) {
  const float y = __builtin_amdgcn_rcpf(r2f);
  return fmaf(y, fmaf(-r2lo, y, fmaf(-r2f, y, 1.0f)), y);
}

__device__ __forceinline__ void lds_add(long long *p, long long v) {
  atomicAdd(reinterpret_cast<unsigned long long *>(p), static_cast<unsigned long long>(v));
}

// The passes.  kGbFast: FastMode's calcForcesIncludingVacuo, above.
// kGbEnergy: FF_GeneralizedBorn_Still::calcEnergies instead (gbff.cpp:178-183,
// 537-596): the exact GB cross term on every pair within Cutoff, whatever its bond
// order and with no ExpApproxThreshold swap, plus FF_NonBonded::calcEnergies with
// Dielectric = DielectricSolute and energy switching; no forces, no dE/da.
// kGbBorn: calcForces with FastMode off (gbff.cpp:186-196): FF_NonBonded::
// calcForces with Dielectric = DielectricSolute and energy switching, and the cross
// term of calcBornForces (gbff.cpp:1189-1345) on every pair within Cutoff, with
// 1/r in place of 1/f_GB (and no dE/da) where uGB <= ExpApproxThreshold.
enum { kGbFast = 0, kGbEnergy = 1, kGbBorn = 2, kGbRadii = 3, kGbChain = 4 };

// Sums of a pass per atom: forces x, y, z and dE/da (pair), Gpol (radii), forces (chain).
constexpr int gb_sums(int pass) { return pass == kGbRadii ? 1 : (pass == kGbChain ? 3 : (pass == kGbEnergy ? 0 : 4)); }

// One workgroup of SPLIT wavefronts per task: one or two i tiles against a run of j
// tiles.  The wavefronts share the staged j tile and take its chunks of 16 steps in
// turn.  Per-pair FP32 arithmetic; FP32 sums over a chunk, fixed point beyond it; the
// energies FP32 over 8 steps, then FP64.
template <int PASS, int SPLIT>
__global__ __launch_bounds__(64 * SPLIT) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_gb_pass(GBPassArgs A) {
  constexpr int NS = gb_sums(PASS);
  constexpr bool PAIR = PASS == kGbFast || PASS == kGbEnergy || PASS == kGbBorn;
  constexpr int T = 64 * SPLIT;
  const GBK K = A.K;
  // the j tile: far loops read the records at lane + t < 128 (each atom twice, no
  // wrap), near loops the FP64 positions and two records at (lane + t) & 63
  __shared__ __align__(16) union Stage {
    struct {
      float4 a[2 * kTile];  // x, y, z (about the tiles' midpoint) and q | V | V
      float2 b[2 * kTile];  // LJ radius, sqrt(eps) | - | W, -
    } far;
    struct {
      double x[kTile], y[kTile], z[kTile];
      float2 p01[kTile], p23[kTile], ia[kTile];  // q, LJ radius, sqrt(eps), a | R, V | R, V, W; 1 / a
    } near;
  } st;
  __shared__ long long jacc[NS > 0 ? NS : 1][kTile], iacc[2][NS > 0 ? NS : 1][kTile];
  __shared__ double es[SPLIT][3];
  const GBTask w = A.tasks[blockIdx.x];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;

  // An atom's position and parameters; a pad (i < 0) has zero parameters and sits far
  // from everything.  Read again for each tile pair: kept, they would cost the loops
  // the registers that let four wavefronts share a SIMD.
  struct Atom {
    double x, y, z;
    float p0, p1, p2, p3;  // q, LJ radius, sqrt(eps), a | R, V | R, V, W
  };
  auto atom = [&](int i, double pad) __attribute__((always_inline)) {
    Atom P{pad, pad, pad, 0.0f, 0.0f, 0.0f, 1.0f};
    if (i >= 0) {
      P.x = A.x[i];
      P.y = A.y[i];
      P.z = A.z[i];
      if (PAIR) {
        P.p0 = A.q[i];
        P.p1 = A.ljr[i];
        P.p2 = A.lje[i];
        P.p3 = A.bornf[i];
      } else {
        P.p0 = A.gbrad[i];
        P.p1 = A.Vj[i];
        if (PASS == kGbChain) P.p2 = chain_weight(A.born, A.deda_in, i, K.P4);
      }
    }
    return P;
  };
  auto lane_atom = [&](int tile) __attribute__((always_inline)) {
    const int2 at = A.tile_atoms[tile];
    return lane < at.y ? at.x + lane : -1;
  };
  for (int k = tid; k < 2 * NS * kTile; k += T) (&iacc[0][0][0])[k] = 0;
  double epol = 0.0, evdw = 0.0, eel = 0.0, efar = 0.0;  // eel: without econv / eps_solute
  // dE/da carries premul, Gpol P4: applied in FP64 as a chunk goes to fixed point
  const double scale_d = K.premul_d, scale_g = (double)K.P4;
  auto sum_of = [&](int c) { return c == 0 ? A.s0 : (c == 1 ? A.s1 : (c == 2 ? A.s2 : A.s3)); };
  // A chunk's sums of one kind to fixed point.  scale * v + 1.5 2^52 holds round(scale v)
  // in its low bits while |scale v| < 2^51: two FP64 instructions a value against seven,
  // and the constant leaves with one subtraction; larger sums (atoms on top of each
  // other) take the long way.
  auto scale_of = [&](int c) {
    return (PASS == kGbRadii ? scale_g : (PAIR && c == 3 ? scale_d : 1.0)) * kFixScale;
  };
  auto to_fix = [&](int c, float v, bool big) __attribute__((always_inline)) -> long long {
    if (big) return fix_from_double((double)v * (scale_of(c) / kFixScale));
    constexpr double kMagic = 6755399441055744.0;
    return __double_as_longlong(fma((double)v, scale_of(c), kMagic)) - __double_as_longlong(kMagic);
  };
  // wave-uniform: some sum of the chunk is too large (or not a number) for the short way
  auto any_big = [&](float m) __attribute__((always_inline)) { return __ballot(!(m < K.fix_lim)) != 0ull; };

  for (int tj = w.tj; tj < w.tj + w.nj; tj++) {
    // ---- what the geometry of the tile pairs allows ---------------------------------
    const GBTile B = A.tiles[tj];
    bool far[2] = {false, false}, inside[2] = {false, false}, live[2] = {false, false};
#pragma unroll
    for (int m = 0; m < 2; m++) {
      if (m >= w.ni) continue;
      const GBTile &C = A.tiles[w.ti + m];
      // FP32 from here on: the margins (1e-3 A and 1e-4 of the distances) are far wider
      // than its rounding
      const float dx = (float)(C.x - B.x), dy = (float)(C.y - B.y), dz = (float)(C.z - B.z);
      const float d = __builtin_amdgcn_sqrtf(dx * dx + dy * dy + dz * dz);
      const float rb = (float)B.rad, reach = (float)C.rad + rb + 1e-3f;
      // every pair's distance is within [lo, hi]
      const float lo = d * (1.0f - 1e-4f) - reach, hi = d * (1.0f + 1e-4f) + reach;
      inside[m] = hi < K.inside;
      live[m] = !(lo > K.outside);
      if (PASS == kGbEnergy || PASS == kGbBorn || w.code >= 0 || !inside[m]) continue;
      // Far: each i atom lies beyond the short-range reach of every j atom, by its
      // distance from the j tile's sphere.  Pair pass: uGB = -r^2 / 4 a_i a_j <=
      // threshold; radii and chain: r^2 / (Ri + Rj)^2 > 1 / P5, where CCF is 1.
      const int i = lane_atom(w.ti + m);
      bool beyond = true;
      if (i >= 0) {
        const float ex = (float)(A.x[i] - B.x), ey = (float)(A.y[i] - B.y), ez = (float)(A.z[i] - B.z);
        const float e = __builtin_amdgcn_sqrtf(ex * ex + ey * ey + ez * ez);
        float need;
        if (PAIR) {
          const float a = A.bornf[i];
          need = a > 0.0f ? __builtin_amdgcn_sqrtf(K.far_k * a * B.amax) : 1e30f;
        } else {
          need = K.far_k * (A.gbrad[i] + B.rmax);
        }
        beyond = e * (1.0f - 1e-4f) > need + rb + 1e-3f;
      }
      far[m] = (!PAIR || K.thresh < 0.0f) && __ballot(!beyond) == 0ull;
    }
    const bool both = far[0] && far[1];
    __syncthreads();  // the previous tile's sums are flushed, its stage is read
    for (int k = tid; k < NS * kTile; k += T) (&jacc[0][0])[k] = 0;
    // the chunks of a tile pair; a diagonal one ends at step 32
    const int nch = tj == w.ti ? 3 : kTile / kChunk;

    // ---- the far loop over a j tile: one i tile or both ------------------------------
    auto far_loop = [&](auto ni_c, int m0, double ox, double oy, double oz) __attribute__((always_inline)) {
      constexpr int NI = decltype(ni_c)::value;  // m0 (uniform): the i tile when it is one
      float px[NI], py[NI], pz[NI], p0[NI], p1[NI], p2[NI];
#pragma unroll
      for (int n = 0; n < NI; n++) {
        const Atom P = atom(lane_atom(w.ti + (NI == 2 ? n : m0)), 5.0e3);
        px[n] = (float)(P.x - ox);
        py[n] = (float)(P.y - oy);
        pz[n] = (float)(P.z - oz);
        p0[n] = PAIR ? P.p0 * K.ec_out : P.p0;
        p1[n] = P.p1;
        p2[n] = P.p2;
      }
      for (int c = wv; c < nch; c += SPLIT) {
      float fx[NI], fy[NI], fz[NI];
      float ax = 0.0f, ay = 0.0f, az = 0.0f;
#pragma unroll
      for (int n = 0; n < NI; n++) fx[n] = fy[n] = fz[n] = 0.0f;
      const int base = lane + c * kChunk;
      for (int h = 0; h < kChunk; h += 8) {
        float ev8 = 0.0f, el8 = 0.0f;
#pragma unroll 2
        for (int u = 0; u < 8; u++) {
          const float4 a = st.far.a[base + h + u];
          float2 b = make_float2(0.0f, 0.0f);
          if (PASS != kGbRadii) b = st.far.b[base + h + u];
          float gx = 0.0f, gy = 0.0f, gz = 0.0f;
#pragma unroll
          for (int n = 0; n < NI; n++) {
            const float dx = px[n] - a.x, dy = py[n] - a.y, dz = pz[n] - a.z;
            const float r2 = dx * dx + dy * dy + dz * dz;
            float g;
            if (PASS == kGbRadii) {
              const float v = __builtin_amdgcn_rcpf(r2 * r2);
              fx[n] = fmaf(v, a.w, fx[n]);
              gx = n == 0 ? v * p1[n] : fmaf(v, p1[n], gx);
              continue;
            } else if (PASS == kGbChain) {
              // -(gpi dE/da_i P4 Vj + gpj dE/da_j P4 Vi) 4 / r^6
              g = -4.0f * fmaf(p2[n], a.w, b.x * p1[n]) * __builtin_amdgcn_rcpf(r2 * r2 * r2);
            } else {
              const float rinv = __builtin_amdgcn_rsqf(r2);
              const float ri2 = rinv * rinv;
              const float e = p0[n] * a.w * rinv;
              const float s = (p1[n] + b.x) * rinv;
              const float s2 = s * s;
              const float Bq = s2 * s2 * s2;
              const float eB = p2[n] * b.y * Bq;
              const float v = fmaf(eB, Bq, -eB);  // eps (B^2 - B)
              el8 += e;
              ev8 += v - eB;
              g = -fmaf(12.0f, v, e) * ri2;
            }
            fx[n] = fmaf(-g, dx, fx[n]);
            fy[n] = fmaf(-g, dy, fy[n]);
            fz[n] = fmaf(-g, dz, fz[n]);
            gx = n == 0 ? g * dx : fmaf(g, dx, gx);
            gy = n == 0 ? g * dy : fmaf(g, dy, gy);
            gz = n == 0 ? g * dz : fmaf(g, dz, gz);
          }
          ax = rotate1(ax) + gx;
          if (PASS != kGbRadii) {
            ay = rotate1(ay) + gy;
            az = rotate1(az) + gz;
          }
        }
        if (PAIR) {
          evdw += (double)ev8;
          efar += (double)el8;
        }
      }
      const int jj = (base + kChunk - 1) & (kTile - 1);
      const float s_j[3] = {ax, ay, az};
      float big = 0.0f;
#pragma unroll
      for (int k = 0; k < (NS >= 3 ? 3 : 1); k++) {
        big = fmax_nan(big, s_j[k]);
#pragma unroll
        for (int n = 0; n < NI; n++) big = fmax_nan(big, k == 0 ? fx[n] : (k == 1 ? fy[n] : fz[n]));
      }
      auto flush = [&](bool slow) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < (NS >= 3 ? 3 : 1); k++) {
          lds_add(&jacc[k][jj], to_fix(k, s_j[k], slow));
#pragma unroll
          for (int n = 0; n < NI; n++)
            lds_add(&iacc[NI == 2 ? n : m0][k][lane], to_fix(k, k == 0 ? fx[n] : (k == 1 ? fy[n] : fz[n]), slow));
        }
      };
      if (any_big(big))
        flush(true);
      else
        flush(false);
      }
    };

    // ---- the near loop: one i tile ----------------------------------------------------
    auto near_loop = [&](auto coded_c, auto inside_c, int m) __attribute__((always_inline)) {
      constexpr bool CODED = decltype(coded_c)::value, IN = decltype(inside_c)::value;
      const Atom P = atom(lane_atom(w.ti + m), 5.0e3);
      const double qx = P.x, qy = P.y, qz = P.z;
      const float p0 = P.p0, p1 = P.p1, p2 = P.p2, p3 = P.p3;
      const float quarter = 0.25f / p3;
      for (int c = wv; c < nch; c += SPLIT) {
      unsigned cw = CODED ? A.codes[((size_t)w.code * (kTile / kChunk) + c) * kTile + lane] : 0u;
      float fx = 0.0f, fy = 0.0f, fz = 0.0f, fd = 0.0f, ax = 0.0f, ay = 0.0f, az = 0.0f, ad = 0.0f;
      for (int h = 0; h < kChunk; h += 8) {
        float ep8 = 0.0f, ev8 = 0.0f, el8 = 0.0f;
        // two steps at a time: the arithmetic of two pairs overlaps, and the short-range
        // part of the pass, which few steps need, is behind one branch for the wavefront
#pragma unroll 1
        for (int u2 = 0; u2 < 8; u2 += 2) {
          double r2d[2];
          float dx[2], dy[2], dz[2], r2f[2];
          float2 a01[2], a23[2], aia[2];
          bool on[2], on_gb[2], nb[2], s14[2], lj[2];
#pragma unroll
          for (int v = 0; v < 2; v++) {
            const int jj = (lane + c * kChunk + h + u2 + v) & (kTile - 1);
            const unsigned code = CODED ? cw & 3u : (unsigned)kPairPlain;
            if (CODED) cw >>= 2;
            const bool valid = !CODED || code != kPairNone;
            double r2 = 0.0;
            {
#pragma clang fp contract(off)
              const double ex = qx - st.near.x[jj], ey = qy - st.near.y[jj], ez = qz - st.near.z[jj];
              if (PAIR || !IN) r2 = ex * ex + ey * ey + ez * ez;  // PD's expression (gbff.cpp:455, 1588-1591)
              dx[v] = (float)ex;
              dy[v] = (float)ey;
              dz[v] = (float)ez;
            }
            r2f[v] = !PAIR && IN ? dx[v] * dx[v] + dy[v] * dy[v] + dz[v] * dz[v] : (float)r2;
            a01[v] = st.near.p01[jj];
            if (PASS != kGbRadii) a23[v] = st.near.p23[jj];
            r2d[v] = r2;
            if (PAIR) {
              aia[v] = st.near.ia[jj];
              on[v] = valid && (IN || r2 <= K.cut2);
              // calcBornEnergy's test on the distance (gbff.cpp:560)
              on_gb[v] = PASS == kGbEnergy ? valid && (IN || r2 < K.gb_lim) : on[v];
              // vdW and Coulomb only for non-bonded and 1-4 pairs
              nb[v] = on[v] && (!CODED || code < kPairBonded);
              s14[v] = CODED && code == kPair14;
              lj[v] = nb[v] && (IN || r2 < K.vdw_lim);  // Dist_ij < VdwCutoff (gbff.cpp:1686)
              if (!(on[v] || on_gb[v])) r2d[v] = r2f[v] = 1.0f;
            } else {
              // only non-bonded and 1-4 partners (gbff.cpp:460-461)
              on[v] = (!CODED || code < kPairBonded) && (IN || r2 <= K.still2);
              r2f[v] = on[v] ? r2f[v] : 1.0f;
            }
          }
          if (!PAIR) {
            // CCF = (0.5 - 0.5 cos th)^2 = sin(th/2)^4 with th = pi P5 r^2 / (Ri + Rj)^2,
            // dccf = 2 (0.5 - 0.5 cos th) sin th th; 1 and 0 beyond r^2 / (Ri + Rj)^2 = 1 / P5
            float rdivR[2], ccf[2], f4[2];  // f4: 4 CCF - dccf
#pragma unroll
            for (int v = 0; v < 2; v++) {
              const float Rs = p0 + a01[v].x;
              rdivR[v] = r2f[v] * __builtin_amdgcn_rcpf(Rs * Rs);
              ccf[v] = 1.0f;
              f4[v] = 4.0f;
            }
            if (__ballot(rdivR[0] <= K.invP5 || rdivR[1] <= K.invP5) != 0ull) {
#pragma unroll
              for (int v = 0; v < 2; v++) {
                const bool close = rdivR[v] <= K.invP5;
                const float hf = close ? rdivR[v] * K.half_pi_P5 : 0.0f;
                const float sn = sin_quarter(hf);
                const float s3 = sn * sn * sn;
                ccf[v] = close ? s3 * sn : 1.0f;
                if (PASS == kGbChain) f4[v] = fmaf(4.0f, ccf[v], -8.0f * hf * s3 * cos_quarter(hf));
              }
            }
#pragma unroll
            for (int v = 0; v < 2; v++) {
              if (PASS == kGbRadii) {
                const float e = on[v] ? ccf[v] * __builtin_amdgcn_rcpf(r2f[v] * r2f[v]) : 0.0f;
                fx = fmaf(e, a01[v].y, fx);
                ax = rotate1(ax) + e * p1;
              } else {
                // both directions of the pair: gpi deda_i P4 Vj + gpj deda_j P4 Vi
                const float g = on[v] ? -fmaf(p2, a01[v].y, a23[v].x * p1) * f4[v] *
                                            __builtin_amdgcn_rcpf(r2f[v] * r2f[v] * r2f[v])
                                      : 0.0f;
                fx = fmaf(-g, dx[v], fx);
                fy = fmaf(-g, dy[v], fy);
                fz = fmaf(-g, dz[v], fz);
                ax = rotate1(ax) + g * dx[v];
                ay = rotate1(ay) + g * dy[v];
                az = rotate1(az) + g * dz[v];
              }
            }
          } else {
            float rinv[2], r[2], qq[2], uGB[2], dS[2], Sw[2];
            // ep, dal: without premul; gg: (dE/dr) / r of the cross term without premul
            float ep[2], dal[2], gg[2], ratio[2];
            bool close[2], edge[2];
#pragma unroll
            for (int v = 0; v < 2; v++) {
              rinv[v] = __builtin_amdgcn_rsqf(r2f[v]);
              r[v] = r2f[v] * rinv[v];
              qq[v] = (PASS == kGbEnergy || on[v]) ? p0 * a01[v].x : 0.0f;
              uGB[v] = -r2f[v] * (quarter * aia[v].x);
              close[v] = PASS == kGbEnergy ? on_gb[v] : on[v] && uGB[v] > K.thresh;
              edge[v] = PASS != kGbEnergy && on[v] && fabsf(uGB[v] - K.thresh) < K.edge;
              ep[v] = dal[v] = gg[v] = 0.0f;
              // switching (r >= InnerCutoff), gbff.cpp:1640-1651; none inside
              dS[v] = 0.0f;
              Sw[v] = 1.0f;
              if (!IN) {
                const float t = fmaxf(r[v] - K.inner, 0.0f);
                const float S0 = 1.0f - (K.invw * t) * (K.invw * t);
                dS[v] = -K.invw2_4 * t * S0;
                Sw[v] = S0 * S0;
              }
            }
            // a pair at the threshold (where the terms jump) is decided in FP64, as PD does
            if (PASS != kGbEnergy && __builtin_expect(__ballot(edge[0] || edge[1]) != 0ull, 0)) {
              const int at = A.tile_atoms[tj].x, i = lane_atom(w.ti + m);
#pragma unroll
              for (int v = 0; v < 2; v++)
                if (edge[v]) {
                  const int jj = (lane + c * kChunk + h + u2 + v) & (kTile - 1);
                  close[v] = -r2d[v] * 0.25 / (A.born[i] * A.born[at + jj]) > (double)K.thresh;
                }
            }
            if (PASS != kGbFast || __ballot(close[0] || close[1]) != 0ull) {
#pragma unroll
              for (int v = 0; v < 2; v++) {
                const float aiaj = p3 * a23[v].y;
                if (PASS == kGbEnergy) {
                  ep[v] = close[v] ? qq[v] * __builtin_amdgcn_rsqf(r2f[v] + aiaj * __expf(uGB[v])) * Sw[v] : 0.0f;
                } else {
                  // 1 / f_GB, 1 ulp; kGbBorn: 1 / r beyond the threshold (tg = 0 gives it)
                  const float tg = close[v] ? __expf(uGB[v]) : 0.0f;
                  const float f = __builtin_amdgcn_rsqf(fmaf(tg, aiaj, r2f[v]));
                  const float e0 = (close[v] || PASS == kGbBorn) ? qq[v] * f : 0.0f;
                  const float el = e0 * (f * f);
                  gg[v] = -el * fmaf(-0.25f, tg, 1.0f);
                  dal[v] = -el * tg * (1.0f - uGB[v]);
                  dal[v] = close[v] ? dal[v] : 0.0f;
                  ep[v] = e0;
                  if (!IN) {
                    gg[v] = fmaf(Sw[v], gg[v], dS[v] * e0 * rinv[v]);
                    dal[v] *= Sw[v];
                    ep[v] *= Sw[v];
                  }
                }
              }
            }
#pragma unroll
            for (int v = 0; v < 2; v++) {
              const float ri2 = rcp_near(r2f[v], (float)(r2d[v] - (double)r2f[v]));
              // eps_solvent where FastMode drops the GB term
              ratio[v] = PASS == kGbFast && !close[v] ? K.ec_ratio : 1.0f;
              // Ee, Fe: without econv / eps_solute; Fe, Fv: (dE/dr) / r
              const float e1 = nb[v] ? qq[v] * (s14[v] ? K.elec14 : 1.0f) * rinv[v] * ratio[v] : 0.0f;
              float Ee = e1, Fe = -e1 * ri2;
              if (!IN) {
                Fe = fmaf(Sw[v], Fe, dS[v] * e1 * rinv[v]);
                Ee *= Sw[v];
              }
              const float eps = (s14[v] ? K.vdw14 : 1.0f) * p2 * a23[v].x;
              const float s = p1 + a01[v].y;
              const float s2 = s * s * ri2;
              const float Bq = s2 * s2 * s2;
              const float eB = lj[v] ? eps * Bq : 0.0f;
              const float w2 = fmaf(eB, Bq, -eB);
              float Ev = w2 - eB, Fv = -12.0f * w2 * ri2;
              if (!IN) {
                const float t = fmaxf(r[v] - K.vdwinner, 0.0f);
                const float V0 = 1.0f - (K.vinvw * t) * (K.vinvw * t);
                const float vdS = -K.vinvw2_4 * t * V0;
                const float VS = V0 * V0;
                Fv = fmaf(VS, Fv, Ev * vdS * rinv[v]);
                Ev *= VS;
              }
              ep8 += ep[v];
              ev8 += Ev;
              el8 += Ee;
              if (PASS == kGbEnergy) continue;
              // along d = p_i - p_j: twice the cross term, vdW and Coulomb
              const float g = fmaf(K.premul2, gg[v], fmaf(K.ec_in, Fe, Fv));
              fd = fmaf(dal[v], a23[v].y, fd);
              ad = rotate1(ad) + dal[v] * p3;
              fx = fmaf(-g, dx[v], fx);
              fy = fmaf(-g, dy[v], fy);
              fz = fmaf(-g, dz[v], fz);
              ax = rotate1(ax) + g * dx[v];
              ay = rotate1(ay) + g * dy[v];
              az = rotate1(az) + g * dz[v];
            }
          }
        }
        if (PAIR) {
          epol += (double)ep8;
          evdw += (double)ev8;
          eel += (double)el8;
        }
      }
      if constexpr (NS > 0) {
        const int jj = (lane + c * kChunk + kChunk - 1) & (kTile - 1);
        const float s_i[4] = {fx, fy, fz, fd}, s_j[4] = {ax, ay, az, ad};
        float big = 0.0f;
#pragma unroll
        for (int k = 0; k < NS; k++) big = fmax_nan(fmax_nan(big, s_i[k]), s_j[k]);
        auto flush = [&](bool slow) __attribute__((always_inline)) {
#pragma unroll
          for (int k = 0; k < NS; k++) {
            lds_add(&jacc[k][jj], to_fix(k, s_j[k], slow));
            lds_add(&iacc[m][k][lane], to_fix(k, s_i[k], slow));
          }
        };
        if (any_big(big))
          flush(true);
        else
          flush(false);
      }
      }
    };

    auto stage_far = [&](double ox, double oy, double oz) {
      if (wv == 0) {
        const Atom P = atom(lane_atom(tj), -5.0e3);
        const float4 a =
            make_float4((float)(P.x - ox), (float)(P.y - oy), (float)(P.z - oz), PAIR ? P.p0 : P.p1);
        const float2 b = PAIR ? make_float2(P.p1, P.p2) : make_float2(P.p2, 0.0f);
        st.far.a[lane] = a;
        st.far.a[lane + kTile] = a;
        if (PASS != kGbRadii) {
          st.far.b[lane] = b;
          st.far.b[lane + kTile] = b;
        }
      }
    };
    if (both) {
      const GBTile C0 = A.tiles[w.ti], C1 = A.tiles[w.ti + 1];
      const double ox = 0.25 * (C0.x + C1.x) + 0.5 * B.x, oy = 0.25 * (C0.y + C1.y) + 0.5 * B.y,
                   oz = 0.25 * (C0.z + C1.z) + 0.5 * B.z;
      stage_far(ox, oy, oz);
      __syncthreads();
      far_loop(std::integral_constant<int, 2>{}, 0, ox, oy, oz);
    } else {
      for (int m = 0; m < w.ni; m++) {
        const bool in = m ? inside[1] : inside[0];
        if (!(m ? live[1] : live[0])) continue;  // uniform over the workgroup
        if (m == 1) __syncthreads();             // the first tile's stage is read
        if (m ? far[1] : far[0]) {
          const GBTile C = A.tiles[w.ti + m];
          const double ox = 0.5 * (C.x + B.x), oy = 0.5 * (C.y + B.y), oz = 0.5 * (C.z + B.z);
          stage_far(ox, oy, oz);
          __syncthreads();
          far_loop(std::integral_constant<int, 1>{}, m, ox, oy, oz);
          continue;
        }
        if (wv == 0) {
          const Atom P = atom(lane_atom(tj), -5.0e3);
          st.near.x[lane] = P.x;
          st.near.y[lane] = P.y;
          st.near.z[lane] = P.z;
          st.near.p01[lane] = make_float2(P.p0, P.p1);
          if (PASS != kGbRadii) st.near.p23[lane] = make_float2(P.p2, P.p3);
          if (PAIR) st.near.ia[lane] = make_float2(1.0f / P.p3, 0.0f);
        }
        __syncthreads();
        if (w.code >= 0)
          in ? near_loop(std::true_type{}, std::true_type{}, m) : near_loop(std::true_type{}, std::false_type{}, m);
        else
          in ? near_loop(std::false_type{}, std::true_type{}, m) : near_loop(std::false_type{}, std::false_type{}, m);
      }
    }
    if constexpr (NS > 0) {  // this j tile's sums
      __syncthreads();
      const int j = lane_atom(tj);
      for (int c = wv; c < NS; c += SPLIT) {
        const long long v = jacc[c][lane];
        if (j >= 0 && v != 0) fix_add(&sum_of(c)[j], v);
      }
    }
  }
  if constexpr (NS > 0) {  // the i tiles' sums (the last barrier above follows every add)
    for (int k = wv; k < w.ni * NS; k += SPLIT) {
      const int m = k / NS, c = k % NS;
      const int i = lane_atom(w.ti + m);
      const long long v = iacc[m][c][lane];
      if (i >= 0 && v != 0) fix_add(&sum_of(c)[i], v);
    }
  }
  if (PAIR) {
    const double sp = wave_sum(epol), sv = wave_sum(evdw), sl = wave_sum(K.ec_in_d * eel + efar);
    if (lane == 0) {
      es[wv][0] = sp;
      es[wv][1] = sv;
      es[wv][2] = sl;
    }
    __syncthreads();
    if (tid == 0) {
      double e3[3] = {0.0, 0.0, 0.0};
      for (int k = 0; k < SPLIT; k++)
        for (int c = 0; c < 3; c++) e3[c] += es[k][c];
      // PD adds each cross term twice (gbff.cpp:1655-1658)
      A.e_part[4 * (size_t)w.slot + 0] = 2.0 * scale_d * e3[0];
      A.e_part[4 * (size_t)w.slot + 1] = e3[1];
      A.e_part[4 * (size_t)w.slot + 2] = e3[2];
      A.e_part[4 * (size_t)w.slot + 3] = 0.0;
    }
  }
}


// ---- the plain comparator ---------------------------------------------------------
// The straightforward single-system GPU form of the FastMode passes, kept as the
// baseline the tiled kernels are measured against: one thread per atom i over
// every other atom j of the system, FP64 arithmetic and FP64 sums per atom (each
// pair evaluated from both sides), no tiles, no LDS; the per-atom force is added
// to the fixed-point accumulator once.  Same physics and pair tests as above.
__global__ __launch_bounds__(256) void k_plain_radii(PlainGB P, const double *__restrict__ x,
                                                     const double *__restrict__ y, const double *__restrict__ z,
                                                     const double *__restrict__ gr, const double *__restrict__ vj,
                                                     const double *__restrict__ q, const double *__restrict__ t123,
                                                     const int8_t *__restrict__ band, const int *__restrict__ sp_off,
                                                     const int *__restrict__ sp_part, const int *__restrict__ sp_ord,
                                                     double *__restrict__ born, float *__restrict__ bornf,
                                                     double *__restrict__ deda, double *__restrict__ eself) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.n) return;
  double g = 0.0;
  for (int j = 0; j < P.n; j++) {
    if (j == i) continue;
    const double dx = x[i] - x[j], dy = y[i] - y[j], dz = z[i] - z[j];
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (r2 > P.still2) continue;
    if (gb_bond_order(i, j, P.mid, band, sp_off, sp_part, sp_ord) <= 2) continue;
    const double Rs = gr[i] + gr[j];
    const double rdivR = r2 / (Rs * Rs);
    double ccf = 1.0;
    if (rdivR <= P.invP5) {
      const double c = 0.5 - 0.5 * cos(rdivR * P.P5 * P.pi);
      ccf = c * c;
    }
    g += P.P4 * vj[j] * ccf / (r2 * r2);
  }
  const double a = -P.halfeconv / (t123[i] + g) + P.offset;
  born[i] = a;
  bornf[i] = (float)a;
  const double ep = P.premul * q[i] * q[i] / a;
  eself[i] = ep;
  deda[i] = -ep / a;
}

__global__ __launch_bounds__(256) void k_plain_pair(PlainGB P, const double *__restrict__ x,
                                                    const double *__restrict__ y, const double *__restrict__ z,
                                                    const double *__restrict__ q, const double *__restrict__ ljr,
                                                    const double *__restrict__ lje, const double *__restrict__ born,
                                                    const int8_t *__restrict__ band, const int *__restrict__ sp_off,
                                                    const int *__restrict__ sp_part, const int *__restrict__ sp_ord,
                                                    long long *__restrict__ fx, long long *__restrict__ fy,
                                                    long long *__restrict__ fz, double *__restrict__ deda,
                                                    double *__restrict__ e3) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.n) return;
  const double ai = born[i];
  double fi[3] = {0.0, 0.0, 0.0}, dai = 0.0, ecross = 0.0, evdw = 0.0, eel = 0.0;
  for (int j = 0; j < P.n; j++) {
    if (j == i) continue;
    const double dx = x[i] - x[j], dy = y[i] - y[j], dz = z[i] - z[j];
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (r2 > P.cut2) continue;
    const int bo = gb_bond_order(i, j, P.mid, band, sp_off, sp_part, sp_ord);
    const double r = sqrt(r2), ir = 1.0 / r;
    const double aj = born[j], aiaj = ai * aj, qq = q[i] * q[j];
    const double u = -r2 * 0.25 / aiaj;
    const double s14e = bo == 3 ? P.elec14 : 1.0;
    const bool nb = bo >= 3;
    double S = 1.0, dS = 0.0;
    if (r >= P.inner) {
      const double t = P.invw * (r - P.inner);
      const double S0 = 1.0 - t * t;
      dS = -4.0 * P.invw * P.invw * (r - P.inner) * S0;
      S = S0 * S0;
    }
    double ep = 0.0, dedr = 0.0, dal = 0.0, Eel = 0.0, Fel = 0.0;
    if (u > P.thresh) {
      const double tg = exp(u);
      const double l = 1.0 / (r2 + tg * aiaj);
      const double f = sqrt(l);
      ep = P.premul * qq * f;
      dedr = -ep * (r - 0.25 * r * tg) * l;
      dal = -ep * tg * (1.0 - u) * l;
      if (nb) {
        Eel = P.ec_in * s14e * qq * ir;
        Fel = -Eel * ir;
      }
      dedr = S * dedr + dS * ep;
      dal *= S;
      ep *= S;
    } else if (nb) {
      Eel = P.ec_out * s14e * qq * ir;
      Fel = -Eel * ir;
    }
    Fel = S * Fel + Eel * dS;
    Eel *= S;
    double Ev = 0.0, Fv = 0.0;
    if (nb && r < P.vdwcut) {
      const double eps = (bo == 3 ? P.vdw14 : 1.0) * lje[i] * lje[j];
      double B = (ljr[i] + ljr[j]) * ir;
      B = B * B;
      B = B * B * B;
      const double A = B * B;
      Ev = eps * (A - 2.0 * B);
      Fv = -12.0 * eps * ir * (A - B);
      if (r > P.vdwinner) {
        const double t = P.vinvw * (r - P.vdwinner);
        const double V0 = 1.0 - t * t;
        const double vdS = -4.0 * P.vinvw * P.vinvw * (r - P.vdwinner) * V0;
        Fv = V0 * V0 * Fv + Ev * vdS;
        Ev *= V0 * V0;
      }
    }
    const double g = (2.0 * dedr + Fv + Fel) * ir;
    fi[0] -= g * dx;
    fi[1] -= g * dy;
    fi[2] -= g * dz;
    dai += dal * aj;
    ecross += ep;
    evdw += 0.5 * Ev;
    eel += 0.5 * Eel;
  }
  fix_add(&fx[i], fix_from_double(fi[0]));
  fix_add(&fy[i], fix_from_double(fi[1]));
  fix_add(&fz[i], fix_from_double(fi[2]));
  deda[i] += dai;
  e3[i] = ecross;
  e3[P.n + i] = evdw;
  e3[2 * P.n + i] = eel;
}

__global__ __launch_bounds__(256) void k_plain_chain(PlainGB P, const double *__restrict__ x,
                                                     const double *__restrict__ y, const double *__restrict__ z,
                                                     const double *__restrict__ gr, const double *__restrict__ vj,
                                                     const double *__restrict__ born, const double *__restrict__ deda,
                                                     const int8_t *__restrict__ band, const int *__restrict__ sp_off,
                                                     const int *__restrict__ sp_part, const int *__restrict__ sp_ord,
                                                     long long *__restrict__ fx, long long *__restrict__ fy,
                                                     long long *__restrict__ fz) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.n) return;
  // w_i = gpi dE/da_i P4, gpi = a_i^2 / 166.0 (gbff.cpp:1772)
  const double wi = (born[i] * born[i] / 166.0) * deda[i] * P.P4;
  double fi[3] = {0.0, 0.0, 0.0};
  for (int j = 0; j < P.n; j++) {
    if (j == i) continue;
    const double dx = x[j] - x[i], dy = y[j] - y[i], dz = z[j] - z[i];
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (r2 > P.still2) continue;
    if (gb_bond_order(i, j, P.mid, band, sp_off, sp_part, sp_ord) <= 2) continue;
    const double Rs = gr[i] + gr[j];
    const double rdivR = r2 / (Rs * Rs);
    double ccf = 1.0, dccf = 0.0;
    if (rdivR <= P.invP5) {
      const double th = rdivR * P.P5 * P.pi;
      const double sq = 0.5 - 0.5 * cos(th);
      ccf = sq * sq;
      dccf = 2.0 * sq * sin(th) * th;
    }
    const double wj = (born[j] * born[j] / 166.0) * deda[j] * P.P4;
    const double dedr = (wi * vj[j] + wj * vj[i]) * (4.0 * ccf - dccf) / (r2 * r2 * r2);
    fi[0] -= dedr * dx;  // dE/dp_i gets dedr (p_j - p_i); the force is its negative
    fi[1] -= dedr * dy;
    fi[2] -= dedr * dz;
  }
  fix_add(&fx[i], fix_from_double(fi[0]));
  fix_add(&fy[i], fix_from_double(fi[1]));
  fix_add(&fz[i], fix_from_double(fi[2]));
}

// Per-system sum of a per-atom array into slot out_off of the system's output.
__global__ void k_seg_sum_atoms(const double *__restrict__ v, const int *__restrict__ first,
                                const int *__restrict__ count, double *__restrict__ out, int out_stride,
                                int out_off) {
  __shared__ double s[256];
  const int sysi = blockIdx.x;
  double a = 0.0;
  for (int k = threadIdx.x; k < count[sysi]; k += 256) a += v[first[sysi] + k];
  s[threadIdx.x] = a;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[(size_t)sysi * out_stride + out_off] = s[0];
}

// A GB evaluation's energies in a launch of their own: block (s, k) takes system s's.
__global__ __launch_bounds__(256) void k_gb_sums(GBSums G) {
  __shared__ double s[4][256];
  gb_sums_block(G, blockIdx.x, blockIdx.y, s);
}

}  // namespace

// ---------------------------------------------------------------------------------------
// Host side.  GBState holds the device arrays of one or more systems concatenated.

GBState::~GBState() = default;

// FF_GeneralizedBorn_Still::calcFixedBornRadiiTerms (gbff.cpp:324-398), FP64 on the host.
void gb_fixed_terms(int n, const double *gbrad, const pdgpu_gb_params &p, const int32_t *off12,
                    const int32_t *idx12, const double *d12, const int32_t *off13, const int32_t *idx13,
                    const double *d13, std::vector<double> &Vj, std::vector<double> &terms123) {
  const double PI = Consts::PI, FourPI = 4.0 * PI;
  auto sqr = [](double v) { return v * v; };
  Vj.assign(n, 0.0);
  terms123.assign(n, 0.0);
  for (int j = 0; j < n; j++) {
    double Rj = gbrad[j];
    if (Rj <= 0.01) Rj = 1.15;  // Qiu et al. radius for hydrogens (gbff.cpp:343-344)
    Vj[j] = FourPI * Rj * Rj * Rj / 3;
    for (int nk = off12[j]; nk < off12[j + 1]; nk++) {
      const int k = idx12[nk];
      double Rk = gbrad[k];
      if (Rk <= 0.01) Rk = 1.15;
      const double rjk = 1.01 * d12[nk];
      const double hjk = Rj * (1.0 + (sqr(Rk) - sqr(Rj) - sqr(rjk)) / (2.0 * Rj * rjk));
      Vj[j] -= PI * sqr(hjk) * (3 * Rj - hjk) / 3;
    }
    if (Vj[j] < 0) Vj[j] = 0;
  }
  for (int i = 0; i < n; i++) {
    double Rj = gbrad[i];
    if (Rj <= 0.01) Rj = 1.15;
    const double term1 = -166.0 / (Rj + p.DielectricOffset + p.P1);
    double term2 = 0;
    for (int nj = off12[i]; nj < off12[i + 1]; nj++)
      term2 += p.P2 * Vj[idx12[nj]] / (sqr(d12[nj]) * sqr(d12[nj]));
    double term3 = 0;
    for (int nj = off13[i]; nj < off13[i + 1]; nj++)
      term3 += p.P3 * Vj[idx13[nj]] / (sqr(d13[nj]) * sqr(d13[nj]));
    terms123[i] = term1 + term2 + term3;
  }
}

void GBState::set_params(const pdgpu_gb_params &p) {
  prm = p;
  const double ec = Consts::econv();
  GBK k{};
  k.cut2 = p.Cutoff * p.Cutoff;
  k.cut = p.Cutoff;
  k.still2 = p.GbsaStillCutoff * p.GbsaStillCutoff;
  // PD compares rounded distances: sqrt(r2) < VdwCutoff and (calcBornEnergy)
  // sqrt(r2) <= Cutoff.  The rounded square root never decreases, so each test is
  // r2 below one FP64 value, found here.
  auto first_at = [](double c, auto beyond) {
    double v = c * c;
    while (!beyond(std::sqrt(v))) v = std::nextafter(v, HUGE_VAL);
    while (v > 0.0 && beyond(std::sqrt(std::nextafter(v, 0.0)))) v = std::nextafter(v, 0.0);
    return v;
  };
  k.vdw_lim = p.VdwCutoff > 0.0 ? first_at(p.VdwCutoff, [&](double r) { return r >= p.VdwCutoff; }) : 0.0;
  k.gb_lim = p.Cutoff >= 0.0 ? first_at(p.Cutoff, [&](double r) { return r > p.Cutoff; }) : 0.0;
  k.premul_d = -Consts::halfeconv() * (1 / p.DielectricSolute - 1 / p.DielectricSolvent);
  k.ec_in_d = ec / p.DielectricSolute;
  k.premul2 = (float)(2.0 * k.premul_d);
  k.ec_in = (float)k.ec_in_d;
  k.ec_out = (float)(ec / p.DielectricSolvent);
  k.ec_ratio = (float)(p.DielectricSolute / p.DielectricSolvent);
  const double w = p.Cutoff - p.InnerCutoff;
  k.inner = (float)p.InnerCutoff;
  k.invw = w > 0 ? (float)(1.0 / w) : 0.0f;
  k.invw2_4 = w > 0 ? (float)(4.0 / (w * w)) : 0.0f;
  const double vw = p.VdwCutoff - p.VdwInnerCutoff;
  k.vdwinner = (float)p.VdwInnerCutoff;
  k.vinvw = vw > 0 ? (float)(1.0 / vw) : 0.0f;
  k.vinvw2_4 = vw > 0 ? (float)(4.0 / (vw * vw)) : 0.0f;
  k.thresh = (float)p.ExpApproxThreshold;
  k.P4 = (float)p.P4;
  k.invP5 = (float)(1 / p.P5);
  k.half_pi_P5 = (float)(0.5 * Consts::PI * p.P5);
  k.vdw14 = (float)p.Vdw14Scaling;
  k.elec14 = (float)p.Elec14Scaling;
  // the passes' geometry tests (k_gb_pass), for the pair pass and for radii / chain: a tile
  // pair inside every cutoff and switching radius, one beyond the cutoff, and the reach
  // of the short-range part (of sqrt(a_i a_j), of Ri + Rj)
  kp = kr = k;
  kp.inside = std::min(std::min((float)std::sqrt(k.cut2), (float)std::sqrt(k.vdw_lim)), std::min(k.inner, k.vdwinner)) - 1e-3f;
  // a chunk sum up to here stays below 2^51 in fixed point, its factor (premul, P4) included
  kp.fix_lim = (float)(4.0e5 / std::max(1.0, std::fabs(k.premul_d)));
  kr.fix_lim = (float)(4.0e5 / std::max(1.0, std::fabs((double)k.P4)));
  kp.edge = 4e-6f * std::max(1.0f, std::fabs(k.thresh));  // FP32's error of uGB is below 1e-6 of it
  kp.outside = (float)p.Cutoff + 1e-3f;
  kp.far_k = -4.0f * k.thresh * (1.0f + 1e-3f);
  kr.inside = (float)p.GbsaStillCutoff - 1e-3f;
  kr.outside = (float)p.GbsaStillCutoff + 1e-3f;
  kr.far_k = std::sqrt(k.invP5) * (1.0f + 1e-3f);
}

// Adds one system (atoms [first, first+count) of the concatenated arrays) and
// its tiles; the tasks are made from all systems in upload().
void GBState::add_system(int first, int count, int mid, const std::vector<int8_t> &band_sys,
                         const std::vector<int> &spi, const std::vector<int> &spj, const std::vector<int> &spo) {
  GBSys S{};
  S.first = first;
  S.count = count;
  S.mid = mid;
  S.band_off = (long)h_band.size();
  S.sp_base = (int)h_sp_off.size();
  h_band.insert(h_band.end(), band_sys.begin(), band_sys.end());
  // sparse partners keyed by the lower local index, last one of a pair wins
  std::vector<int> cnt(count + 1, 0);
  for (size_t k = 0; k < spi.size(); k++) cnt[std::min(spi[k], spj[k]) + 1]++;
  for (int i = 0; i < count; i++) cnt[i + 1] += cnt[i];
  const int part_base = (int)h_sp_part.size();
  std::vector<int> fill(cnt.begin(), cnt.end() - 1);
  h_sp_part.resize(part_base + spi.size());
  h_sp_ord.resize(part_base + spi.size());
  const int nt = (count + kTile - 1) / kTile;
  std::vector<std::pair<int, int>> linked;  // tile pairs that hold a sparse partner
  for (size_t k = 0; k < spi.size(); k++) {
    const int lo = std::min(spi[k], spj[k]), hi = std::max(spi[k], spj[k]);
    h_sp_part[part_base + fill[lo]] = hi;
    h_sp_ord[part_base + fill[lo]] = spo[k];
    fill[lo]++;
    linked.emplace_back(lo / kTile, hi / kTile);
  }
  std::sort(linked.begin(), linked.end());
  h_linked.push_back(std::move(linked));
  for (int i = 0; i <= count; i++) h_sp_off.push_back(part_base + cnt[i]);
  h_sys.push_back(S);
  h_tile_beg.push_back((int)h_tile_atoms.size());
  for (int t = 0; t < nt; t++) h_tile_atoms.push_back(make_int2(first + t * kTile, std::min(kTile, count - t * kTile)));
  n_atoms_total = std::max(n_atoms_total, first + count);
}

// The tasks of every system.  A tile pair whose bond orders can differ from 7 (and
// every diagonal one) is a task with codes; the others are taken two i tiles (2a,
// 2a + 1) at a time against runs of j tiles.  A longer run shares the i tiles' sums and
// the task's opening over more j tiles but leaves fewer tasks.  Pair pass at runs of
// 1 / 2 / 3 / 4 (each at its best split): 54,560 tile pairs 287 / 277 / 274 / 281 us,
// 13,640 90 / 92 / 92 / 92, 8,704 83 / 78 / 92 / 80, 3,160 30 / 32 / 38 / 46.  Heavier
// tasks come first, so the light ones fill the end.
void GBState::make_tasks() {
  h_tasks.clear();
  h_coded.clear();
  h_slot_beg.clear();
  h_slot_end.clear();
  long units = 0;
  for (size_t s = 0; s < h_sys.size(); s++) {
    const long nt = (h_sys[s].count + kTile - 1) / kTile;
    units += nt * (nt + 1) / 2;
  }
  const int run = units >= 32768 ? 3 : (units >= 8192 ? 2 : 1);
  int slot = 0, codes = 0;
  for (size_t s = 0; s < h_sys.size(); s++) {
    const int nt = (h_sys[s].count + kTile - 1) / kTile, base = h_tile_beg[s], mid = h_sys[s].mid;
    auto coded = [&](int ti, int tj) {
      return (tj - ti) * kTile - (kTile - 1) < mid ||  // the smallest j - i over the tile pair
             std::binary_search(h_linked[s].begin(), h_linked[s].end(), std::make_pair(ti, tj));
    };
    h_slot_beg.push_back(slot);
    auto push = [&](int ti, int ni, int tj, int nj, bool with_codes) {
      h_tasks.push_back(GBTask{(int)s, base + ti, ni, base + tj, nj, with_codes ? codes++ : -1, slot++, 0});
    };
    for (int a = 0; a < nt; a += 2) {
      for (int m = 0; m < 2; m++)
        for (int tj = a + m; a + m < nt && tj < nt; tj++)
          if (coded(a + m, tj)) push(a + m, 1, tj, 1, true);
      // the i tiles that take j tile tj without codes: 0 none, 1 the first, 2 the second, 3 both
      auto takes = [&](int tj) {
        return (tj > a && !coded(a, tj) ? 1 : 0) | (a + 1 < nt && tj > a + 1 && !coded(a + 1, tj) ? 2 : 0);
      };
      for (int tj = a + 1; tj < nt;) {
        const int who = takes(tj);
        int nj = 1;
        while (nj < run && tj + nj < nt && takes(tj + nj) == who) nj++;
        if (who) push(who == 2 ? a + 1 : a, who == 3 ? 2 : 1, tj, nj, false);
        tj += nj;
      }
    }
    h_slot_end.push_back(slot);
  }
  n_slots = slot;
  auto weight = [](const GBTask &w) { return w.code >= 0 ? 3 : 2 * w.ni * w.nj; };
  std::stable_sort(h_tasks.begin(), h_tasks.end(),
                   [&](const GBTask &a, const GBTask &b) { return weight(a) > weight(b); });
  for (size_t k = 0; k < h_tasks.size(); k++)
    if (h_tasks[k].code >= 0) h_coded.push_back((int)k);
}

namespace {
// The autotuner's choices for the process, by (atoms, systems, FastMode): a
// GB state of the same shape starts with the split tuned for it.
std::mutex g_split_mutex;
std::map<std::tuple<int, int, int>, std::array<int, 3>> g_split_choice;
std::tuple<int, int, int> split_key(const GBState &G) {
  return std::make_tuple(G.n_atoms_total, (int)G.h_sys.size(), G.prm.FastMode ? 1 : 0);
}
}  // namespace

void GBState::upload(hipStream_t s) {
  {
    std::lock_guard<std::mutex> lk(g_split_mutex);
    auto it = g_split_choice.find(split_key(*this));
    if (it != g_split_choice.end())
      for (int k = 0; k < 3; k++) split[k] = it->second[k];
  }
  make_tasks();
  tasks.upload(h_tasks, s);
  sysd.upload(h_sys.data(), h_sys.size(), s);
  tile_atoms.upload(h_tile_atoms, s);
  tiles.resize(h_tile_atoms.size());
  if (h_band.empty()) h_band.push_back(7);
  band.upload(h_band, s);
  sp_off.upload(h_sp_off, s);
  if (h_sp_part.empty()) {
    h_sp_part.push_back(0);
    h_sp_ord.push_back(0);
  }
  sp_part.upload(h_sp_part, s);
  sp_ord.upload(h_sp_ord, s);
  slot_beg.upload(h_slot_beg, s);
  slot_end.upload(h_slot_end, s);
  std::vector<int> f, c;
  for (auto &S : h_sys) {
    f.push_back(S.first);
    c.push_back(S.count);
  }
  sys_first.upload(f, s);
  sys_count.upload(c, s);
  const int n = n_atoms_total;
  gpol.resize(n);
  deda.resize(n);
  born.resize(n);
  bornf.resize(n);
  eself.resize(n);
  e_part.resize((size_t)n_slots * 4);
  coded.upload(h_coded, s);
  codes.resize(h_coded.size() * (kTile / kChunk) * kTile);
  hipLaunchKernelGGL(k_gb_codes, dim3((unsigned)h_coded.size()), dim3(64), 0, s, tasks.p, coded.p, tile_atoms.p,
                     sysd.p, band.p, sp_off.p, sp_part.p, sp_ord.p, codes.p);
  PDGPU_HIP(hipGetLastError());
}

// A pass's launch: every task at `split` wavefronts, or (0) at the number that fills
// the chip: a task's chunks follow each other in one wavefront, so few tasks leave
// SIMDs idle, while many pay for each wavefront's share of the opening.  Radii / pair
// / chain at splits 1, 2, 4: 1,700 tasks 22 / 44 / 32, 16 / 33 / 25, 14 / 30 / 22 us; 4,000
// tasks 39 / 88 / 59, 31 / 78 / 46, 34 / 82 / 48; 21,000 tasks 101 / 274 / 171, 113 / 302 /
// 187, 153 / 346 / 213.
template <int PASS>
void GBState::launch_pass(hipStream_t s, const GBPassArgs &A, int sp) {
  const unsigned nt = (unsigned)h_tasks.size();
  if (sp == 0) sp = nt < 3072 ? 4 : (nt < 12288 ? 2 : 1);
  if (sp == 4)
    hipLaunchKernelGGL((k_gb_pass<PASS, 4>), dim3(nt), dim3(256), 0, s, A);
  else if (sp == 2)
    hipLaunchKernelGGL((k_gb_pass<PASS, 2>), dim3(nt), dim3(128), 0, s, A);
  else
    hipLaunchKernelGGL((k_gb_pass<PASS, 1>), dim3(nt), dim3(64), 0, s, A);
}

GBPassArgs GBState::pass_args(const double *x, const double *y, const double *z, long long *fx, long long *fy,
                              long long *fz) const {
  GBPassArgs A{};
  A.K = kp;
  A.tasks = tasks.p;
  A.tile_atoms = tile_atoms.p;
  A.tiles = tiles.p;
  A.codes = codes.p;
  A.x = x;
  A.y = y;
  A.z = z;
  A.q = q.p;
  A.ljr = ljr.p;
  A.lje = lje.p;
  A.bornf = bornf.p;
  A.gbrad = gbrad.p;
  A.Vj = Vj.p;
  A.born = born.p;
  A.deda_in = deda.p;
  A.s0 = fx;
  A.s1 = fy;
  A.s2 = fz;
  A.s3 = deda.p;
  A.e_part = e_part.p;
  return A;
}

PlainGB GBState::plain_args() const {
  PlainGB P{};
  P.n = n_atoms_total;
  P.mid = h_sys.empty() ? 0 : h_sys[0].mid;
  P.still2 = prm.GbsaStillCutoff * prm.GbsaStillCutoff;
  P.cut2 = prm.Cutoff * prm.Cutoff;
  P.vdwcut = prm.VdwCutoff;
  P.inner = prm.InnerCutoff;
  P.vdwinner = prm.VdwInnerCutoff;
  P.invw = prm.Cutoff > prm.InnerCutoff ? 1.0 / (prm.Cutoff - prm.InnerCutoff) : 0.0;
  P.vinvw = prm.VdwCutoff > prm.VdwInnerCutoff ? 1.0 / (prm.VdwCutoff - prm.VdwInnerCutoff) : 0.0;
  P.premul = -Consts::halfeconv() * (1 / prm.DielectricSolute - 1 / prm.DielectricSolvent);
  P.ec_in = Consts::econv() / prm.DielectricSolute;
  P.ec_out = Consts::econv() / prm.DielectricSolvent;
  P.thresh = prm.ExpApproxThreshold;
  P.P4 = prm.P4;
  P.P5 = prm.P5;
  P.invP5 = 1 / prm.P5;
  P.vdw14 = prm.Vdw14Scaling;
  P.elec14 = prm.Elec14Scaling;
  P.halfeconv = Consts::halfeconv();
  P.offset = prm.BornRadiusOffset;
  P.pi = Consts::PI;
  return P;
}

void GBState::set_split(const int32_t *s3) {
  for (int k = 0; k < 3; k++) {
    const int v = s3 ? s3[k] : 1;
    if (v != 1 && v != 2 && v != 4) throw EngineError(PDGPU_ERR_ARG, "GB split must be 1, 2 or 4");
    split[k] = v;
  }
}

// Runs the three passes.  Forces are added to fx/fy/fz (fixed point, kcal/mol/A);
// per-system energies (kcal/mol) go to out[s*stride + off + {0: pol cross, 1: vdw,
// 2: elec, 3: -}] and out[s*stride + off + 4] (pol self).  open: what shares the opening
// launch; the plain comparator takes nothing along.
void GBState::run(hipStream_t s, const double *x, const double *y, const double *z, long long *fx, long long *fy,
                  long long *fz, double *out, int out_stride, int out_off, Engine *timer_owner, bool energy_only,
                  const GBOpen *open, bool sums) {
  const int n = n_atoms_total;
  const int nsys = (int)h_sys.size();
  if (plain) {
    if (energy_only || !prm.FastMode || nsys != 1)
      throw EngineError(PDGPU_ERR_ARG, "the plain GB comparator runs one system's FastMode forces");
    const PlainGB P = plain_args();
    const int g = (n + 255) / 256;
    {
      ScopedTimerOpt t(timer_owner, "gb_radii");
      hipLaunchKernelGGL(k_plain_radii, dim3(g), dim3(256), 0, s, P, x, y, z, pl_gr.p, pl_vj.p, pl_q.p, terms123.p,
                         band.p, sp_off.p, sp_part.p, sp_ord.p, born.p, bornf.p, pl_deda.p, eself.p);
    }
    {
      ScopedTimerOpt t(timer_owner, "gb_pair");
      hipLaunchKernelGGL(k_plain_pair, dim3(g), dim3(256), 0, s, P, x, y, z, pl_q.p, pl_r.p, pl_e.p, born.p, band.p,
                         sp_off.p, sp_part.p, sp_ord.p, fx, fy, fz, pl_deda.p, pl_e3.p);
    }
    {
      ScopedTimerOpt t(timer_owner, "gb_chain");
      hipLaunchKernelGGL(k_plain_chain, dim3(g), dim3(256), 0, s, P, x, y, z, pl_gr.p, pl_vj.p, born.p, pl_deda.p,
                         band.p, sp_off.p, sp_part.p, sp_ord.p, fx, fy, fz);
    }
    PDGPU_HIP(hipGetLastError());
    for (int c = 0; c < 3; c++)
      hipLaunchKernelGGL(k_seg_sum_atoms, dim3(1), dim3(256), 0, s, pl_e3.p + (size_t)c * n, sys_first.p,
                         sys_count.p, out, out_stride, out_off + c);
    hipLaunchKernelGGL(k_seg_sum_atoms, dim3(1), dim3(256), 0, s, eself.p, sys_first.p, sys_count.p, out,
                       out_stride, out_off + 4);
    return;
  }
  const GBPassArgs A = pass_args(x, y, z, fx, fy, fz);
  const int ntiles = (int)h_tile_atoms.size();
  const dim3 tg((ntiles + 3) / 4);
  const GBOpen none{}, &O = open ? *open : none;
  const SumList L = O.sums ? *O.sums : SumList{};
  hipLaunchKernelGGL(k_gb_open, dim3(O.bonded_blocks + tg.x + (L.n > 0 || L.record ? 1 : 0)), dim3(256), 0, s, ntiles,
                     tile_atoms.p, x, y, z, gbrad.p, tiles.p, gpol.p, O.bonded, O.bonded_blocks, fx, fy, fz,
                     O.bonded_partial, O.bonded_eterm, L);
  {
    ScopedTimerOpt t(timer_owner, "gb_radii");
    GBPassArgs R = A;
    R.K = kr;
    R.s0 = gpol.p;
    launch_pass<kGbRadii>(s, R, split[0]);
  }
  hipLaunchKernelGGL(k_gb_finalize_radii, tg, dim3(256), 0, s, ntiles, tile_atoms.p, Consts::halfeconv(),
                     prm.BornRadiusOffset, kp.premul_d, terms123.p, gpol.p, q.p, born.p, bornf.p, deda.p, eself.p,
                     tiles.p);
  {
    ScopedTimerOpt t(timer_owner, "gb_pair");
    if (energy_only)
      launch_pass<kGbEnergy>(s, A, split[1]);
    else if (prm.FastMode)
      launch_pass<kGbFast>(s, A, split[1]);
    else
      launch_pass<kGbBorn>(s, A, split[1]);
  }
  if (!energy_only) {
    ScopedTimerOpt t(timer_owner, "gb_chain");
    GBPassArgs C = A;
    C.K = kr;
    launch_pass<kGbChain>(s, C, split[2]);
  }
  PDGPU_HIP(hipGetLastError());
  if (sums) hipLaunchKernelGGL(k_gb_sums, dim3(nsys, 2), dim3(256), 0, s, sum_args(out, out_stride, out_off));
}

// The tile kernels' inputs (radii, dE/da, chain weights) come from one full pass
// first; each kernel then runs kTuneLaunches times at every split.  The force and
// dE/da accumulators are left modified: a full evaluation must follow.
void GBState::autotune(hipStream_t s, const double *x, const double *y, const double *z, long long *fx,
                       long long *fy, long long *fz, double *out, int out_stride, int out_off, double *us) {
  constexpr int kTuneLaunches = 5;
  run(s, x, y, z, fx, fy, fz, out, out_stride, out_off, nullptr, false);
  hipEvent_t a, b;
  PDGPU_HIP(hipEventCreate(&a));
  PDGPU_HIP(hipEventCreate(&b));
  const GBPassArgs A = pass_args(x, y, z, fx, fy, fz);
  GBPassArgs R = A, Q = A;
  R.K = Q.K = kr;
  R.s0 = gpol.p;
  for (int k = 0; k < 3; k++) {
    double best = 1e300;
    int best_split = 1;
    for (int m = 0; m < 3; m++) {
      const int sp = 1 << m;
      auto launch = [&]() {
        if (k == 0)
          launch_pass<kGbRadii>(s, R, sp);
        else if (k == 1 && prm.FastMode)
          launch_pass<kGbFast>(s, A, sp);
        else if (k == 1)
          launch_pass<kGbBorn>(s, A, sp);
        else
          launch_pass<kGbChain>(s, Q, sp);
      };
      launch();  // warm
      PDGPU_HIP(hipEventRecord(a, s));
      for (int r = 0; r < kTuneLaunches; r++) launch();
      PDGPU_HIP(hipEventRecord(b, s));
      PDGPU_HIP(hipEventSynchronize(b));
      float ms = 0.0f;
      PDGPU_HIP(hipEventElapsedTime(&ms, a, b));
      const double t = 1e3 * (double)ms / kTuneLaunches;
      if (us) us[3 * k + m] = t;
      if (t < best) {
        best = t;
        best_split = sp;
      }
    }
    split[k] = best_split;
  }
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  PDGPU_HIP(hipGetLastError());
  std::lock_guard<std::mutex> lk(g_split_mutex);
  g_split_choice[split_key(*this)] = {split[0], split[1], split[2]};
}

// ---- single-system glue ------------------------------------------------------------

void Engine::launch_gb(double *energy_slots, bool energy_only, double *bonded_slots, bool sums) {
  require(have_gb, "GB component not set up");
  // gbff.cpp takes every distance as p_j - p_i with no image: GB is a vacuum model
  require(!periodic, "GB runs in vacuum: PD's GB takes raw displacements, no periodic images");
  GBOpen O{};
  if (bonded_slots) {
    O.bonded = bonded_arrays();
    O.bonded_blocks = bonded_blocks(nbonds, nangles, ntors);
    // alternating halves: the sums of the step before read the other one
    e_partial_bonded.resize((size_t)O.bonded_blocks * 8);
    O.bonded_partial = e_partial_bonded.p + (size_t)gb_bonded_sel * O.bonded_blocks * 4;
    gb_bonded_sel ^= 1;
  }
  O.sums = &gb_sums;
  gb->run(stream, x.p, y.p, z.p, fbx.p, fby.p, fbz.p, energy_slots, 8, 0, this, energy_only, &O, sums);
  gb_sums = SumList{};
  if (bonded_slots) defer_sum4(O.bonded_partial, O.bonded_blocks, bonded_slots);
}

// h: [0] cross (2x pair sum), [1] vdw, [2] elec, [3] -, [4] self, kcal/mol.  With
// FastMode off, calcForces adds the polarisation energy to epot alone.
void gb_slots_to_energies(const double *h, bool pol_terms, pdgpu_energies &e) {
  const double kj = Consts::kcal_to_J();
  const double pol = h[0] + h[4];
  e.epot_vdw += h[1] * kj;
  e.epot_elec += h[2] * kj;
  if (pol_terms) {
    e.epot_pol += pol * kj;
    e.epot_pol_cross += h[0] * kj;
    e.epot_pol_self += h[4] * kj;
  }
  e.epot += (h[1] + h[2] + pol) * kj;
}

}  // namespace pdgpu

using pdgpu::Engine;

extern "C" int pdgpu_set_gb_split(pdgpu_engine *h, const int32_t *split) {
  return pdgpu::guarded(h, [&](Engine &E) {
    E.require(E.have_gb, "GB component not set up");
    E.gb->set_split(split);
  });
}

extern "C" int pdgpu_set_gb_plain(pdgpu_engine *h, int32_t on) {
  return pdgpu::guarded(h, [&](Engine &E) {
    E.require(E.have_gb, "GB component not set up");
    E.require(!on || E.gb->prm.FastMode, "the plain GB comparator computes FastMode forces");
    E.gb->plain = on != 0;
  });
}

extern "C" int pdgpu_autotune_gb(pdgpu_engine *h, int32_t *split, double *us) {
  return pdgpu::guarded(h, [&](Engine &E) {
    E.require(E.have_gb && E.have_positions, "GB component or positions not set up");
    E.fbx.resize(E.n);
    E.fby.resize(E.n);
    E.fbz.resize(E.n);
    E.e_out.resize(24);
    E.gb->autotune(E.stream, E.x.p, E.y.p, E.z.p, E.fbx.p, E.fby.p, E.fbz.p, E.e_out.p + 8, 8, 0, us);
    E.sync();
    E.last_components = 0;  // the accumulators hold tuning runs, not an evaluation
    if (split)
      for (int k = 0; k < 3; k++) split[k] = E.gb->split[k];
  });
}

extern "C" int pdgpu_setup_gb(pdgpu_engine *h, const pdgpu_gb_params *p, const double *gbradius,
                              const int32_t *off12, const int32_t *idx12, const double *d12, const int32_t *off13,
                              const int32_t *idx13, const double *d13) {
  Engine *E = reinterpret_cast<Engine *>(h);
  if (!E) return PDGPU_ERR_ARG;
  try {
    PDGPU_HIP(hipSetDevice(E->device));
    E->require(p && gbradius && off12 && off13, "null GB argument");
    E->require(!E->h_charge.empty(), "atom parameters not set");
    E->require(p->DielectricSolute > 0 && p->DielectricSolvent > 0 && p->P5 > 0, "bad GB parameters");
    const int n = E->n;
    for (int i = 0; i < n; i++) {
      for (int k = off12[i]; k < off12[i + 1]; k++) E->require(idx12[k] >= 0 && idx12[k] < n, "cov12 index");
      for (int k = off13[i]; k < off13[i + 1]; k++) E->require(idx13[k] >= 0 && idx13[k] < n, "cov13 index");
    }
    std::vector<double> Vj, t123;
    pdgpu::gb_fixed_terms(n, gbradius, *p, off12, idx12, d12, off13, idx13, d13, Vj, t123);
    auto gb = std::make_unique<pdgpu::GBState>();
    gb->set_params(*p);
    gb->add_system(0, n, E->mid, E->h_band, E->h_sp_i, E->h_sp_j, E->h_sp_order);
    gb->upload(E->stream);
    std::vector<float> q(n), r(n), e(n), g(n), v(n);
    const double es = 1.0 / std::sqrt(pdgpu::Consts::kcal_to_J());
    for (int i = 0; i < n; i++) {
      q[i] = (float)E->h_charge[i];
      r[i] = (float)E->h_radius[i];
      e[i] = (float)(E->h_epsilon[i] * es);
      g[i] = (float)gbradius[i];
      v[i] = (float)Vj[i];
    }
    gb->q.upload(q, E->stream);
    gb->ljr.upload(r, E->stream);
    gb->lje.upload(e, E->stream);
    gb->gbrad.upload(g, E->stream);
    gb->Vj.upload(v, E->stream);
    gb->terms123.upload(t123, E->stream);
    {  // FP64 copies for the plain comparator
      std::vector<double> qd(n), rd(n), ed(n), gd(gbradius, gbradius + n);
      for (int i = 0; i < n; i++) {
        qd[i] = E->h_charge[i];
        rd[i] = E->h_radius[i];
        ed[i] = E->h_epsilon[i] * es;
      }
      gb->pl_q.upload(qd, E->stream);
      gb->pl_r.upload(rd, E->stream);
      gb->pl_e.upload(ed, E->stream);
      gb->pl_gr.upload(gd, E->stream);
      gb->pl_vj.upload(Vj, E->stream);
      gb->pl_deda.resize(n);
      gb->pl_e3.resize((size_t)3 * n);
    }
    E->sync();
    E->gb = std::move(gb);
    E->have_gb = true;
    // FF_NonBonded::setup requests the cutoffs; GB also wants the shadow list (gbff.cpp:97-101)
    E->list_cutoff = std::max(E->list_cutoff, std::max(p->Cutoff, p->VdwCutoff));
    return PDGPU_OK;
  } catch (const pdgpu::EngineError &x) {
    E->last_error = x.what();
    return x.code;
  } catch (const std::exception &x) {
    E->last_error = x.what();
    return PDGPU_ERR_ARG;
  }
}

extern "C" int pdgpu_get_born_radii(pdgpu_engine *h, double *radii) {
  Engine *E = reinterpret_cast<Engine *>(h);
  if (!E || !radii) return PDGPU_ERR_ARG;
  if (!E->have_gb) {
    E->last_error = "GB component not set up";
    return PDGPU_ERR_ARG;
  }
  try {
    E->gb->born.download(radii, E->n, E->stream);
    E->sync();
    return PDGPU_OK;
  } catch (const pdgpu::EngineError &x) {
    E->last_error = x.what();
    return x.code;
  }
}
