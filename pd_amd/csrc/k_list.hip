// k_list.hip -- WorkSpace::cleanSpace + NeighbourList::calcNewList on the device.
//
// PD builds the list with an O(N^2) double loop (neighbourlist.cpp:336-439 for
// PeriodicBox, 247-333 for InfiniteSpace).  Here atoms are binned into grid
// columns, sorted by z inside each column and cut into clusters of 8 slots.
// For every i-cluster one wavefront finds the j-clusters (index >= i-cluster)
// whose bounding boxes come within Cutoff+Padding, then tests every atom pair
// with PD's own FP64 arithmetic: d = p_j - p_i, wrapped by the `while` minimum-
// image loops that also produce the image number, r^2 = (x*x + y*y) + z*z with
// no FMA, kept when r^2 <= (Cutoff+Padding)^2.  The result is the exact PD pair
// set, stored per i-cluster as 8-byte entries:
//   x: j slot (24 bits) | image (5 bits) << 24 | (j atom has an LJ epsilon) << 29
//      (image as seen from the i atom)
//   y: listed mask over the 8 i atoms (8 bits) | 2-bit bond-order code per i atom
//      << 8 (0 = order 7, 1 = 1-2, 2 = 1-3, 3 = 1-4) | rank of the j atom's
//      cluster in the work group's candidate table << 24
// Bond orders follow the list builder: the band matrix for |i-j| < MaxIndexDelta,
// 7 otherwise, then the off-diagonal corrections (neighbourlist.cpp:179-220).
#include "engine.hpp"

#include <algorithm>
#include <climits>
#include <cmath>

namespace pdgpu {

namespace {

constexpr int kMaxCand = 1536;  // candidate j-clusters per work group (LDS)
constexpr int kCandPart = 512;  // candidates found by one wave of the group
// The candidate table is ordered by the distance of each candidate's box from
// the group's box, in three bands (below 4 A, below 8 A, the rest): the nearest
// candidates hold the most list entries, and the first kGroupRanks of the table
// get LDS accumulators in the nonbonded kernel.
constexpr int kDistBands = 3;
constexpr double kBand1 = 16.0, kBand2 = 64.0;  // squared box distances (A^2)

// Also clears the grid's column counts (ncol of them) for the binning that follows.
__global__ void k_clean_space(int n_mol, const int *__restrict__ first, const int *__restrict__ last,
                              double *__restrict__ x, double *__restrict__ y, double *__restrict__ z,
                              double bx, double by, double bz, int ncol, int *__restrict__ col_count) {
#pragma clang fp contract(off)
  // WorkSpace::cleanSpace (workspace.cpp:371-380); centre of geometry as
  // MoleculeBase::getCentreOfGeometry(ifirst, ilast) (molecule.cpp:850-858).
  int m = blockIdx.x * blockDim.x + threadIdx.x;
  for (int c = m; c < ncol; c += gridDim.x * blockDim.x) col_count[c] = 0;
  if (m >= n_mol) return;
  const double hx = bx / 2.0, hy = by / 2.0, hz = bz / 2.0;
  double cx = 0.0, cy = 0.0, cz = 0.0;
  const int f = first[m], l = last[m];
  for (int i = f; i <= l; i++) {
    cx += x[i];
    cy += y[i];
    cz += z[i];
  }
  const double cnt = (double)(l - f + 1);
  cx /= cnt;
  cy /= cnt;
  cz /= cnt;
  double ix = cx, iy = cy, iz = cz;  // PeriodicBox::getClosestImage (space.h:215-227)
  for (int it = 0; it < 64 && ix > hx; it++) ix -= bx;
  for (int it = 0; it < 64 && ix < -hx; it++) ix += bx;
  for (int it = 0; it < 64 && iy > hy; it++) iy -= by;
  for (int it = 0; it < 64 && iy < -hy; it++) iy += by;
  for (int it = 0; it < 64 && iz > hz; it++) iz -= bz;
  for (int it = 0; it < 64 && iz < -hz; it++) iz += bz;
  const double sx = ix - cx, sy = iy - cy, sz = iz - cz;
  for (int i = f; i <= l; i++) {
    x[i] += sx;
    y[i] += sy;
    z[i] += sz;
  }
}

__global__ void k_bbox(int n, const double *__restrict__ x, const double *__restrict__ y,
                       const double *__restrict__ z, double *__restrict__ out) {
  __shared__ double s[6][1024];
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    lo[0] = fmin(lo[0], x[i]); hi[0] = fmax(hi[0], x[i]);
    lo[1] = fmin(lo[1], y[i]); hi[1] = fmax(hi[1], y[i]);
    lo[2] = fmin(lo[2], z[i]); hi[2] = fmax(hi[2], z[i]);
  }
  for (int d = 0; d < 3; d++) {
    s[d][threadIdx.x] = lo[d];
    s[3 + d][threadIdx.x] = hi[d];
  }
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int d = 0; d < 3; d++) {
        s[d][threadIdx.x] = fmin(s[d][threadIdx.x], s[d][threadIdx.x + w]);
        s[3 + d][threadIdx.x] = fmax(s[3 + d][threadIdx.x], s[3 + d][threadIdx.x + w]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 6) out[threadIdx.x] = s[threadIdx.x][0];
}

struct GridArgs {
  int periodic;
  int ncx, ncy;
  double lo_x, lo_y, w_x, w_y;   // column origin and width
  double L[3];                   // box (periodic)
};

__device__ __forceinline__ double wrap_coord(double v, double L) {
  // representative in [-L/2, L/2) used for binning only
  return v - L * floor(v / L + 0.5);
}

// Adds 1 for every lane to counter[key] with one atomic per distinct key in the
// wave (atoms of a wave are usually neighbours, so their keys mostly agree);
// returns each lane's rank among the lanes that share its key plus the base
// the atomic returned, i.e. a slot unique to the lane.
__device__ __forceinline__ int wave_aggregated_add(int *counter, int key, bool active) {
  const int lane = threadIdx.x & 63;
  unsigned long long pending = __ballot(active);
  int slot = 0;
  while (pending) {  // each round retires at least the leader's key
    const int leader = __ffsll((long long)pending) - 1;
    const int lk = __shfl(key, leader, 64);
    const unsigned long long same = __ballot(active && key == lk) & pending;
    int base = 0;
    if (lane == leader) base = atomicAdd(&counter[lk], __popcll(same));
    base = __shfl(base, leader, 64);
    if ((same >> lane) & 1ull) slot = base + __popcll(same & ((1ull << lane) - 1ull));
    pending &= ~same;
  }
  return slot;
}

__global__ void k_bin(int n, GridArgs g, const double *__restrict__ x, const double *__restrict__ y,
                      const double *__restrict__ z, double *__restrict__ wx, double *__restrict__ wy,
                      double *__restrict__ wz, int *__restrict__ wrap, int *__restrict__ atom_col,
                      int *__restrict__ col_count) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool v = i < n;
  int col = 0;
  if (v) {
    double a = x[i], b = y[i], c = z[i];
    int k[3] = {0, 0, 0};
    if (g.periodic) {
      // wrapped = v + k L with k = -floor(v / L + 1/2): the representative in [-L/2, L/2)
      k[0] = -(int)floor(a / g.L[0] + 0.5);
      k[1] = -(int)floor(b / g.L[1] + 0.5);
      k[2] = -(int)floor(c / g.L[2] + 0.5);
      a = wrap_coord(a, g.L[0]);
      b = wrap_coord(b, g.L[1]);
      c = wrap_coord(c, g.L[2]);
    }
    wx[i] = a;
    wy[i] = b;
    wz[i] = c;
    wrap[i] = (k[0] & 0xFF) | ((k[1] & 0xFF) << 8) | ((k[2] & 0xFF) << 16);
    int cx = (int)floor((a - g.lo_x) / g.w_x);
    int cy = (int)floor((b - g.lo_y) / g.w_y);
    cx = min(max(cx, 0), g.ncx - 1);
    cy = min(max(cy, 0), g.ncy - 1);
    col = cy * g.ncx + cx;
    atom_col[i] = col;
  }
  (void)wave_aggregated_add(col_count, col, v);
}

// Single-workgroup exclusive scans over the columns; then the work groups (the
// clusters of each column cut into runs of kGroup, their work counters cleared),
// the cleared pair-search counters and the cluster count in counter[3] for the
// host's check.
__global__ void k_scan_columns(int ncol, const int *__restrict__ col_count, int *__restrict__ col_atom_start,
                               int *__restrict__ col_cl_start, int *__restrict__ col_ncl,
                               int *__restrict__ col_fill, int *__restrict__ col_grp_start,
                               int *__restrict__ n_clusters, int *__restrict__ n_groups,
                               int *__restrict__ grp_first, int *__restrict__ grp_count,
                               int *__restrict__ grp_work, unsigned long long *__restrict__ counter) {
  __shared__ int sa[1024], sc[1024], sg[1024];
  __shared__ int carry_a, carry_c, carry_g;
  if (threadIdx.x == 0) {
    carry_a = 0;
    carry_c = 0;
    carry_g = 0;
  }
  __syncthreads();
  for (int base = 0; base < ncol; base += 1024) {
    int c = base + threadIdx.x;
    int cnt = c < ncol ? col_count[c] : 0;
    int ncl = (cnt + kClusterSize - 1) / kClusterSize;
    int ngr = (ncl + kGroup - 1) / kGroup;
    sa[threadIdx.x] = cnt;
    sc[threadIdx.x] = ncl;
    sg[threadIdx.x] = ngr;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {  // Hillis-Steele inclusive scan
      int va = threadIdx.x >= (unsigned)off ? sa[threadIdx.x - off] : 0;
      int vc = threadIdx.x >= (unsigned)off ? sc[threadIdx.x - off] : 0;
      int vg = threadIdx.x >= (unsigned)off ? sg[threadIdx.x - off] : 0;
      __syncthreads();
      sa[threadIdx.x] += va;
      sc[threadIdx.x] += vc;
      sg[threadIdx.x] += vg;
      __syncthreads();
    }
    if (c < ncol) {
      const int c0 = carry_c + sc[threadIdx.x] - ncl, g0 = carry_g + sg[threadIdx.x] - ngr;
      col_atom_start[c] = carry_a + sa[threadIdx.x] - cnt;
      col_cl_start[c] = c0;
      col_grp_start[c] = g0;
      col_ncl[c] = ncl;
      col_fill[c] = 0;
      for (int k = 0; k * kGroup < ncl; k++) {
        grp_first[g0 + k] = c0 + k * kGroup;
        grp_count[g0 + k] = min(kGroup, ncl - k * kGroup);
        grp_work[g0 + k] = 0;
      }
    }
    __syncthreads();
    if (threadIdx.x == 1023) {
      carry_a += sa[1023];
      carry_c += sc[1023];
      carry_g += sg[1023];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    *n_clusters = carry_c;
    *n_groups = carry_g;
    counter[0] = 0;
    counter[1] = 0;
    counter[2] = 0;
    counter[3] = (unsigned long long)carry_c;
  }
}

__global__ void k_fill_columns(int n, const int *__restrict__ atom_col, const int *__restrict__ col_atom_start,
                               int *__restrict__ col_fill, int *__restrict__ col_atoms) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool v = i < n;
  const int c = v ? atom_col[i] : 0;
  const int k = wave_aggregated_add(col_fill, c, v);  // order inside a column is fixed by the sort below
  if (v) col_atoms[col_atom_start[c] + k] = i;
}

// Per-slot data for the pair search: the binning's wrapped position, the atom
// index, the wrap counts (one signed byte per axis: wrapped = PD position +
// count * box), whether the atom has sparse bond-order partners (bit 24) and
// whether it has a Lennard-Jones epsilon (bit 25).
struct SlotList {
  double wx, wy, wz;
  int orig, aux;
};

// Rank of each atom inside its column by (wrapped z, atom index): a total order,
// so the slot assignment does not depend on the atomic fill order.  One
// workgroup per column; columns of up to kSortLds atoms are ranked from LDS.
// Then the column's slot records: one thread per slot, the 8 lanes of a
// cluster reducing its bounding box (min/max of the wrapped positions of its
// atoms) with lane exchanges, and (with q) the nonbonded parameters per slot.
constexpr int kSortLds = 2048;
__global__ __launch_bounds__(256) void k_sort_columns(int ncol, const int *__restrict__ col_count,
                                                      const int *__restrict__ col_atom_start,
                                                      const int *__restrict__ col_cl_start,
                                                      const int *__restrict__ col_atoms, const double *__restrict__ wx,
                                                      const double *__restrict__ wy, const double *__restrict__ wz,
                                                      const int *__restrict__ wrap, const int *__restrict__ sp_off,
                                                      const float *__restrict__ lj_eps, const float *__restrict__ q,
                                                      const float *__restrict__ lj_r, const float4 *__restrict__ prm_lo,
                                                      float4 *__restrict__ sprm, float4 *__restrict__ sprm_lo,
                                                      int *__restrict__ slot_orig, int *__restrict__ orig_slot,
                                                      int *__restrict__ cl_col, SlotList *__restrict__ sl,
                                                      double *__restrict__ lo, double *__restrict__ hi) {
  __shared__ double sz[kSortLds];
  __shared__ int sa[kSortLds];
  __shared__ int by_rank[kSortLds];       // position in sa/sz of the atom of each rank | LJ flag << 30
  __shared__ unsigned char slj[kSortLds];  // the atom has an LJ epsilon
  const int c = blockIdx.x;
  if (c >= ncol) return;
  const int s0 = col_atom_start[c], cnt = col_count[c];
  const bool in_lds = cnt <= kSortLds;
  // the unfilled slots of the column's last cluster hold no atom
  if ((int)threadIdx.x < kClusterSize && (cnt & (kClusterSize - 1)) != 0) {
    const int r = (cnt & ~(kClusterSize - 1)) + (int)threadIdx.x;
    if (r >= cnt) slot_orig[col_cl_start[c] * kClusterSize + r] = -1;
  }
  // sort key: z, with NaN as +inf so that the ranks stay a permutation; ties
  // are broken by the atom index
  auto key = [](double z) { return z == z ? z : (double)INFINITY; };
  // the LDS arrays are padded to a multiple of 8 with entries that rank after
  // every atom, so the rank loop reads 8 at a time without bounds tests
  const int cnt8 = (cnt + 7) & ~7;
  if (in_lds)
    for (int k = threadIdx.x; k < cnt8; k += blockDim.x) {
      if (k < cnt) {
        const int a = col_atoms[s0 + k];
        sa[k] = a;
        sz[k] = key(wz[a]);
        slj[k] = (lj_eps == nullptr || lj_eps[a] != 0.0f) ? 1 : 0;
      } else {
        sa[k] = INT_MAX;
        sz[k] = (double)INFINITY;
      }
    }
  __syncthreads();
  for (int k = threadIdx.x; k < cnt; k += blockDim.x) {
    const int a = in_lds ? sa[k] : col_atoms[s0 + k];
    const double za = in_lds ? sz[k] : key(wz[a]);
    int rank = 0;
    if (in_lds) {  // uniform: the common case runs from LDS, 8 entries per step, no branches
      for (int m0 = 0; m0 < cnt8; m0 += 8) {
        double zb[8];
        int ab[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
          zb[u] = sz[m0 + u];
          ab[u] = sa[m0 + u];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) rank += ((zb[u] < za) | ((zb[u] == za) & (ab[u] < a))) ? 1 : 0;
      }
      by_rank[rank] = k | ((int)slj[k] << 30);
    } else {
      for (int m = 0; m < cnt; m++) {
        const int b = col_atoms[s0 + m];
        const double zb = key(wz[b]);
        rank += (zb < za || (zb == za && b < a)) ? 1 : 0;
      }
      const int slot = col_cl_start[c] * kClusterSize + rank;
      slot_orig[slot] = a;
      orig_slot[a] = slot;
      if ((rank & (kClusterSize - 1)) == 0) cl_col[slot / kClusterSize] = c;
    }
  }
  if (in_lds) {  // uniform
  __syncthreads();
  // Inside each cluster of 8 consecutive ranks, the atoms with a Lennard-Jones
  // epsilon come first (in z order), then the others: the nonbonded kernel skips
  // the LJ arithmetic for slots that hold none.
  for (int r = threadIdx.x; r < cnt; r += blockDim.x) {
    const int base = r & ~(kClusterSize - 1), end = min(base + kClusterSize, cnt);
    const int br = by_rank[r];
    const int a = sa[br & 0x3FFFFFFF];
    const bool lj = (br >> 30) != 0;
    int pos = 0, nlj = 0;
#pragma unroll
    for (int q = base; q < base + kClusterSize; q++) {
      const bool lq = q < end && (by_rank[q] >> 30) != 0;
      nlj += lq ? 1 : 0;
      pos += (q < r && lq == lj) ? 1 : 0;
    }
    if (!lj) pos += nlj;
    const int slot = col_cl_start[c] * kClusterSize + base + pos;
    slot_orig[slot] = a;
    orig_slot[a] = slot;
    if (r == base) cl_col[slot / kClusterSize] = c;
  }
  }
  __syncthreads();  // the column's slot_orig entries are written
  const int s0c = col_cl_start[c] * kClusterSize, ns = (cnt + kClusterSize - 1) & ~(kClusterSize - 1);
  for (int r0 = 0; r0 < ns; r0 += blockDim.x) {  // whole clusters of 8 lanes: blockDim is a multiple of 8
    const int r = r0 + (int)threadIdx.x;
    const bool live = r < ns;
    const int s = s0c + r;
    const int a = live ? slot_orig[s] : -1;
    SlotList v;
    if (a >= 0) {
      v.wx = wx[a];
      v.wy = wy[a];
      v.wz = wz[a];
      v.orig = a;
      v.aux = wrap[a] | ((sp_off[a + 1] > sp_off[a]) ? (1 << 24) : 0) |
              ((lj_eps == nullptr || lj_eps[a] != 0.0f) ? (1 << 25) : 0);
    } else {
      v.wx = v.wy = v.wz = 0.0;
      v.orig = -1;
      v.aux = 0;
    }
    if (live) {
      sl[s] = v;
      if (q) {
        const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        sprm[s] = a >= 0 ? make_float4(q[a], lj_r[a], lj_eps[a], 0.0f) : zero;
        sprm_lo[s] = a >= 0 ? prm_lo[a] : zero;
      }
    }
    double l[3] = {a >= 0 ? v.wx : 1e300, a >= 0 ? v.wy : 1e300, a >= 0 ? v.wz : 1e300};
    double h[3] = {a >= 0 ? v.wx : -1e300, a >= 0 ? v.wy : -1e300, a >= 0 ? v.wz : -1e300};
#pragma unroll
    for (int off = 1; off < kClusterSize; off <<= 1)
#pragma unroll
      for (int d = 0; d < 3; d++) {
        l[d] = fmin(l[d], __shfl_xor(l[d], off, 64));
        h[d] = fmax(h[d], __shfl_xor(h[d], off, 64));
      }
    if (live && (s & (kClusterSize - 1)) == 0) {
      const int cl = s / kClusterSize;
      for (int d = 0; d < 3; d++) {
        lo[3 * cl + d] = l[d];
        hi[3 * cl + d] = h[d];
      }
    }
  }
}

__global__ void k_fill_int(int *__restrict__ p, int v, int count) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) p[i] = v;
}


__device__ __forceinline__ int wrap_digit(int aux, int axis) { return (int)(int8_t)((aux >> (8 * axis)) & 0xFF); }
// image index contribution of the wrap counts: 9 kx + 3 ky + kz
__device__ __forceinline__ int wrap_image(int aux) {
  return 9 * wrap_digit(aux, 0) + 3 * wrap_digit(aux, 1) + wrap_digit(aux, 2);
}

struct SearchArgs {
  int periodic;
  int ncx, ncy;
  int Dx, Dy;                   // column search half-widths
  double lo_x, lo_y, w_x, w_y;  // column grid (wrapped frame): column (cx, cy) covers lo + c w .. lo + (c+1) w
  double L[3];
  double half[3];
  double rlist2;                // (Cutoff+Padding)^2, PD's sqrIncludeLimit
  double rlist2_lo, rlist2_hi;  // band around rlist2 resolved with PD's own arithmetic
  double Rbox2;                 // squared bbox pruning radius (rlist plus a margin)
  int fast;                     // every pair inside rlist is its own minimum image
  int mid;                      // BondOrder::m_MaxIndexDelta
  int stride;                   // entries reserved per i-cluster
  int pass, npass;              // this launch takes the stencil cells t with t % npass == pass
};

__device__ __forceinline__ int bond_code(int oa, int ob, bool lo_sparse, int mid, const int8_t *__restrict__ band,
                                         const int *__restrict__ sp_off, const int *__restrict__ sp_part,
                                         const int *__restrict__ sp_ord) {
  int hi = max(oa, ob), lo = min(oa, ob);
  int bo = 7;
  if (hi - lo < mid) bo = band[(long)lo * mid + (hi - lo - 1)];
  // off-diagonal corrections (neighbourlist.cpp:179-220): the last partner entry wins
  if (lo_sparse)
    for (int k = sp_off[lo]; k < sp_off[lo + 1]; k++)
      if (sp_part[k] == hi) bo = sp_ord[k];
  bo &= 7;
  return bo == 1 ? 1 : bo == 2 ? 2 : bo == 3 ? 3 : 0;
}

__device__ __forceinline__ unsigned spread8(unsigned m) {
  m = (m | (m << 4)) & 0x0F0Fu;
  m = (m | (m << 2)) & 0x3333u;
  m = (m | (m << 1)) & 0x5555u;
  return m;
}

__global__ __launch_bounds__(64 * kGroup) void k_pair_search(
    SearchArgs A, const int *__restrict__ n_groups, const int *__restrict__ grp_first,
    const int *__restrict__ grp_count, const int *__restrict__ cl_col, const int *__restrict__ col_cl_start,
    const int *__restrict__ col_ncl, const double *__restrict__ cl_lo, const double *__restrict__ cl_hi,
    const SlotList *__restrict__ sl, const double *__restrict__ px, const double *__restrict__ py,
    const double *__restrict__ pz, const int8_t *__restrict__ band, const int *__restrict__ sp_off,
    const int *__restrict__ sp_part, const int *__restrict__ sp_ord, uint2 *__restrict__ entries,
    int *__restrict__ cl_entry_count, int *__restrict__ wg_ncand, int *__restrict__ wg_cand,
    int *__restrict__ grp_work, unsigned long long *__restrict__ counter) {
#pragma clang fp contract(off)
  // phase 1 fills the two halves with the waves' candidate parts; phase 2
  // reuses the space for each wave's list of candidates near its own cluster
  __shared__ int cand[2 * kGroup * kCandPart];
  __shared__ int join_cl[kMaxCand];
  __shared__ unsigned char join_sh[kMaxCand];
  __shared__ SlotList s_i[kGroup][kClusterSize];
  __shared__ int part_n[kGroup];
  __shared__ int part_nb[kGroup][kDistBands];
  __shared__ int s_ncand, s_over;
  int *const cand_cl = cand, *const cand_sh = cand + kGroup * kCandPart;
  const int g = blockIdx.x;
  if (g >= *n_groups) return;  // the whole workgroup leaves together
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c0 = grp_first[g], ng = grp_count[g];
  double glo[3], ghi[3];  // bounding box of the group's clusters
  for (int d = 0; d < 3; d++) {
    glo[d] = cl_lo[3 * c0 + d];
    ghi[d] = cl_hi[3 * c0 + d];
  }
  for (int k = 1; k < ng; k++)
    for (int d = 0; d < 3; d++) {
      glo[d] = fmin(glo[d], cl_lo[3 * (c0 + k) + d]);
      ghi[d] = fmax(ghi[d], cl_hi[3 * (c0 + k) + d]);
    }
  const int col = cl_col[c0];
  const int cx = col % A.ncx, cy = col / A.ncx;

  // ---- phase 1: candidate j-clusters in a fixed order ------------------------
  // The group's own clusters come first (ranks 0..ng-1), then every cluster of
  // the column stencil, image by image, whose box comes within reach of the
  // group's box.  Only j-clusters >= the group's first cluster are candidates
  // (each unordered cluster pair is searched from its lower cluster).  The
  // stencil cells are dealt to the waves round-robin; each wave fills its own
  // part of the LDS table with each candidate's distance band, and the parts
  // are joined band by band, in wave order within a band.
  // With npass > 1 (a candidate table that did not fit) each launch takes every
  // npass-th cell of the stencil, so its candidates are a disjoint share.
  const int own = A.pass == 0 ? ng : 0;  // the group's own clusters: the first pass only
  {
    const int kz_lo = A.periodic ? -1 : 0, kz_hi = A.periodic ? 1 : 0;
    int nw = 0;  // this wave's candidates
    int *my_cl = cand_cl + wave * kCandPart, *my_sh = cand_sh + wave * kCandPart;
    const int wx = 2 * A.Dx + 1, ncell = (2 * A.Dy + 1) * wx;
    // this wave's stencil cells: first_c, first_c + stride_c, ...; a lane first
    // looks up one cell each (its column, image and z extent, every load of the
    // 64 cells in flight together), then the wave takes the cells' items -- a cluster
    // under a z image -- in order, 64 at a time whatever the cell (a cell holds a few
    // clusters: one at a time, each was a round of its own memory latency; the search of
    // 1,536 atoms 58 -> 48 us, of 98,304 200 -> 193)
    const int stride_c = kGroup * A.npass, first_c = A.pass + wave * A.npass;
    const int nk = first_c < ncell ? (ncell - 1 - first_c) / stride_c + 1 : 0;
    for (int k0 = 0; k0 < nk; k0 += 64) {
      // the cell's items: its clusters from the group's first on, for each z image in reach
      int c_first = 0, c_items = 0;
      unsigned c_pack = 0;  // kx + 1 | (ky + 1) << 2 | z images << 4 | clusters << 8
      if (k0 + lane < nk) {
        const int cell = first_c + (k0 + lane) * stride_c;
        const int dy = cell / wx - A.Dy, dx = cell % wx - A.Dx;
        int uy = cy + dy, ky = 0, ux = cx + dx, kx = 0;
        bool ok = true;
        if (A.periodic) {
          for (int it = 0; it < 4 && uy < 0; it++) { uy += A.ncy; ky -= 1; }
          for (int it = 0; it < 4 && uy >= A.ncy; it++) { uy -= A.ncy; ky += 1; }
          for (int it = 0; it < 4 && ux < 0; it++) { ux += A.ncx; kx -= 1; }
          for (int it = 0; it < 4 && ux >= A.ncx; it++) { ux -= A.ncx; kx += 1; }
          ok = ky >= -1 && ky <= 1 && uy >= 0 && uy < A.ncy && kx >= -1 && kx <= 1 && ux >= 0 && ux < A.ncx;
        } else {
          ok = uy >= 0 && uy < A.ncy && ux >= 0 && ux < A.ncx;
        }
        if (ok) {
          const int jcol = uy * A.ncx + ux;
          const double shx = kx * A.L[0], shy = ky * A.L[1];
          // the whole column (its grid rectangle, widened by 1e-3 A against rounding)
          // out of reach of the group's box: no cluster of it can be a candidate
          const double cx0 = A.lo_x + ux * A.w_x + shx - 1e-3, cx1 = cx0 + A.w_x + 2e-3;
          const double cy0 = A.lo_y + uy * A.w_y + shy - 1e-3, cy1 = cy0 + A.w_y + 2e-3;
          const double gx = fmax(0.0, fmax(cx0 - ghi[0], glo[0] - cx1));
          const double gy = fmax(0.0, fmax(cy0 - ghi[1], glo[1] - cy1));
          if (gx * gx + gy * gy <= A.Rbox2) {
            const int cs = col_cl_start[jcol], nc = col_ncl[jcol];
            c_first = max(cs, c0);
            const int left = cs + nc - c_first;
            if (left > 0) {
              // the column's z extent (its clusters are z-ordered) against each image
              const double zlo = cl_lo[3 * cs + 2], zhi = cl_hi[3 * (cs + nc - 1) + 2];
              unsigned zm = 0;
              for (int kz = kz_lo; kz <= kz_hi; kz++) {
                const double shz = kz * A.L[2];
                const double gz = fmax(0.0, fmax(zlo + shz - ghi[2], glo[2] - (zhi + shz)));
                if (!(gz * gz > A.Rbox2)) zm |= 1u << (kz + 1);
              }
              c_items = left * __popc(zm);
              c_pack = (unsigned)(kx + 1) | (unsigned)(ky + 1) << 2 | zm << 4 | (unsigned)left << 8;
            }
          }
        }
      }
      int c_end = c_items;  // items up to and with this lane's cell
      for (int off = 1; off < 64; off <<= 1) {
        const int v = __shfl_up(c_end, off, 64);
        if (lane >= off) c_end += v;
      }
      const int c_start = c_end - c_items, total = __shfl(c_end, 63, 64);
      for (int i0 = 0; i0 < total; i0 += 64) {
        const int item = i0 + lane;
        int q = 0;  // the lane whose cell holds the item: the first with c_end > item
        for (int half = 32; half >= 1; half >>= 1)
          if (__shfl(c_end, q + half - 1, 64) <= item) q += half;
        const int start = __shfl(c_start, q, 64), first = __shfl(c_first, q, 64);
        const unsigned pack = (unsigned)__shfl((int)c_pack, q, 64);
        bool ok = item < total;
        int cj = 0, sh = 0, band_id = 0;
        if (ok) {
          const int left = (int)(pack >> 8), zi = (item - start) / left;
          unsigned zm = (pack >> 4) & 7u;
          for (int k = 0; k < zi; k++) zm &= zm - 1u;
          const int kx = (int)(pack & 3u) - 1, ky = (int)((pack >> 2) & 3u) - 1, kz = __ffs((int)zm) - 2;
          cj = first + (item - start) - zi * left;
          sh = (kx + 1) * 9 + (ky + 1) * 3 + (kz + 1);
          ok = !(sh == 13 && cj < c0 + ng);
          const double shx = kx * A.L[0], shy = ky * A.L[1], shz = kz * A.L[2];
          const double g0 = fmax(0.0, fmax(cl_lo[3 * cj] + shx - ghi[0], glo[0] - (cl_hi[3 * cj] + shx)));
          const double g1 = fmax(0.0, fmax(cl_lo[3 * cj + 1] + shy - ghi[1], glo[1] - (cl_hi[3 * cj + 1] + shy)));
          const double g2 = fmax(0.0, fmax(cl_lo[3 * cj + 2] + shz - ghi[2], glo[2] - (cl_hi[3 * cj + 2] + shz)));
          const double d2 = g0 * g0 + g1 * g1 + g2 * g2;
          ok = ok && d2 <= A.Rbox2;
          band_id = (d2 > kBand1 ? 1 : 0) + (d2 > kBand2 ? 1 : 0);
        }
        const unsigned long long b = __ballot(ok);
        const int pre = __popcll(b & ((1ull << lane) - 1ull));
        if (ok && nw + pre < kCandPart) {
          my_cl[nw + pre] = cj;
          my_sh[nw + pre] = sh | (band_id << 8);
        }
        nw += __popcll(b);
      }
    }
    if (lane == 0) part_n[wave] = nw;
    // this wave's candidates per distance band (its part is read back by other lanes)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int m = min(nw, kCandPart);
    int nb[kDistBands] = {};
    for (int k0 = 0; k0 < m; k0 += 64) {
      const int bid = k0 + lane < m ? (my_sh[k0 + lane] >> 8) : -1;
#pragma unroll
      for (int q = 0; q < kDistBands; q++) nb[q] += __popcll(__ballot(bid == q));
    }
    if (lane == 0)
      for (int q = 0; q < kDistBands; q++) part_nb[wave][q] = nb[q];
  }
  __syncthreads();
  if (threadIdx.x == 0) {  // join: own clusters, then the waves' parts in order
    int tot = own, over = 0;
    for (int w = 0; w < kGroup; w++) {
      over |= part_n[w] > kCandPart;
      tot += min(part_n[w], kCandPart);
    }
    s_ncand = tot;
    s_over = over || tot > kMaxCand;
  }
  __syncthreads();
  {
    // this wave's start in each band: the own clusters, the nearer bands, then
    // the preceding waves' candidates of the same band
    int off[kDistBands];
    int start = own;
#pragma unroll
    for (int q = 0; q < kDistBands; q++) {
      off[q] = start;
      for (int w = 0; w < kGroup; w++) {
        if (w < wave) off[q] += part_nb[w][q];
        start += part_nb[w][q];
      }
    }
    const int m = min(part_n[wave], kCandPart);
    // move this wave's part into place (a separate join buffer keeps the reads and writes apart)
    for (int k0 = 0; k0 < m; k0 += 64) {
      const int k = k0 + lane;
      const int v = k < m ? cand_sh[wave * kCandPart + k] : -1;
      const int bid = v >= 0 ? (v >> 8) : -1;
#pragma unroll
      for (int q = 0; q < kDistBands; q++) {
        const unsigned long long bq = __ballot(bid == q);
        const int pos = off[q] + __popcll(bq & ((1ull << lane) - 1ull));
        if (bid == q && pos < kMaxCand) {
          join_cl[pos] = cand_cl[wave * kCandPart + k];
          join_sh[pos] = (unsigned char)(v & 0xFF);
        }
        off[q] += __popcll(bq);
      }
    }
    if (wave == 0 && lane < own) {
      join_cl[lane] = c0 + lane;
      join_sh[lane] = 13;
    }
    if (wave < ng && lane < kClusterSize) s_i[wave][lane] = sl[(c0 + wave) * kClusterSize + lane];
  }
  __syncthreads();
  const bool cand_overflow = s_over != 0;
  const int ncand = min(s_ncand, kMaxCand);
  // the candidate table the nonbonded kernel mirrors in LDS (ranks < kGroupRanks),
  // from the first pass; later passes' entries are unranked
  const int nr = min(ncand, kGroupRanks);
  if (A.pass == 0) {
    for (int t = threadIdx.x; t < nr; t += blockDim.x) wg_cand[(size_t)g * kGroupStride + t] = join_cl[t];
    if (threadIdx.x == 0) wg_ncand[g] = nr;
  }
  if (wave >= ng) return;

  // ---- phase 2a: this wave's cluster against the candidates' boxes -----------
  const int ci = c0 + wave;
  constexpr int kNearPerWave = 2 * kCandPart * 2;  // 16-bit slots of the phase-1 space per wave
  static_assert(kNearPerWave >= kMaxCand, "a wave's near list must hold every candidate");
  unsigned short *near = reinterpret_cast<unsigned short *>(cand) + wave * kNearPerWave;
  int nnear = 0;
  {
    const double ilo0 = cl_lo[3 * ci], ilo1 = cl_lo[3 * ci + 1], ilo2 = cl_lo[3 * ci + 2];
    const double ihi0 = cl_hi[3 * ci], ihi1 = cl_hi[3 * ci + 1], ihi2 = cl_hi[3 * ci + 2];
    for (int base = 0; base < ncand; base += 64) {
      const int k = base + lane;
      bool ok = false;
      if (k < ncand) {
        const int cj = join_cl[k];
        if (cj >= ci) {  // searched from the lower cluster
          const int csh = join_sh[k];
          const double shx = (csh / 9 - 1) * A.L[0], shy = ((csh / 3) % 3 - 1) * A.L[1],
                       shz = (csh % 3 - 1) * A.L[2];
          double g0 = fmax(0.0, fmax(cl_lo[3 * cj] + shx - ihi0, ilo0 - (cl_hi[3 * cj] + shx)));
          double g1 = fmax(0.0, fmax(cl_lo[3 * cj + 1] + shy - ihi1, ilo1 - (cl_hi[3 * cj + 1] + shy)));
          double g2 = fmax(0.0, fmax(cl_lo[3 * cj + 2] + shz - ihi2, ilo2 - (cl_hi[3 * cj + 2] + shz)));
          ok = (g0 * g0 + g1 * g1 + g2 * g2) <= A.Rbox2;
        }
      }
      const unsigned long long b = __ballot(ok);
      if (ok) near[nnear + __popcll(b & ((1ull << lane) - 1ull))] = (unsigned short)k;
      nnear += __popcll(b);
    }
  }
  // the list is read back by other lanes of the same wave
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  // ---- phase 2b: exact PD pair tests, lane = (candidate, j atom), loop over i atoms
  // A pair is found through exactly one (cluster, shift) candidate: the one
  // whose shift is PD's minimum image less the difference of the binning's
  // wrap counts.  Pairs clearly inside or outside rlist are decided from the
  // wrapped positions (their rounding error is orders of magnitude below the
  // band); pairs in the band, and every pair of a box too small for the minimum
  // image to be implied, take PD's own arithmetic on its positions.
  uint2 *E = entries + (size_t)ci * A.stride;
  const int jj = lane & 7;
  // A listed pair's image is PD's minimum image, which equals the candidate's
  // shift plus the difference of the two atoms' wrap counts (the exact path
  // below accepts a pair only then), so it is jimg - (the i atom's wrap image).
  // When the cluster's atoms share one wrap image, every lane's pairs share one
  // image and each lane writes at most one entry per round.
  int wimg[kClusterSize];
  bool i_uniform = true;
  // a pair can carry a bond-order code only if its atom indices are less than
  // mid apart or one of the two has sparse partners: the cluster's index span
  // widened by mid bounds the j atoms that need the lookup
  int i_lo = INT_MAX, i_hi = INT_MIN;
  bool i_sparse = false;
  unsigned i_valid = 0;  // the cluster's real (not padding) slots
#pragma unroll
  for (int ii = 0; ii < kClusterSize; ii++) {
    const SlotList li = s_i[wave][ii];
    wimg[ii] = wrap_image(li.aux);
    if (li.orig >= 0) {
      i_valid |= 1u << ii;
      if (wimg[ii] != wrap_image(s_i[wave][0].aux)) i_uniform = false;
      i_lo = min(i_lo, li.orig);
      i_hi = max(i_hi, li.orig);
      i_sparse = i_sparse || ((li.aux >> 24) & 1);
    }
  }
  // later passes append to the entries of the earlier ones
  const int cnt0 = A.pass == 0 ? 0 : __builtin_amdgcn_readfirstlane(cl_entry_count[ci]);
  int cnt = cnt0;
  // the first round's j slot; each round loads the next round's while it tests
  int nk = (lane >> 3) < nnear ? (int)near[lane >> 3] : -1;
  SlotList nlj = sl[(nk >= 0 ? join_cl[nk] : ci) * kClusterSize + jj];
  for (int b0 = 0; b0 < nnear; b0 += 8) {
    const bool have = nk >= 0;
    const int k = have ? nk : 0;
    const int cj = have ? join_cl[k] : ci;
    const int csh = have ? (int)join_sh[k] : 13;
    const SlotList lj = nlj;
    {
      const int t = b0 + 8 + (lane >> 3);
      nk = t < nnear ? (int)near[t] : -1;
      nlj = sl[(nk >= 0 ? join_cl[nk] : ci) * kClusterSize + jj];
    }
    const int sx = csh / 9 - 1, sy = (csh / 3) % 3 - 1, sz = csh % 3 - 1;
    const double shx = sx * A.L[0], shy = sy * A.L[1], shz = sz * A.L[2];
    const int sb = cj * kClusterSize + jj;
    const int ob = lj.orig;
    const double jx = lj.wx + shx, jy = lj.wy + shy, jz = lj.wz + shz;
    const int jimg = 13 + 9 * sx + 3 * sy + sz + wrap_image(lj.aux);
    unsigned lm = 0, codes = 0;
    // The 8 tests without divergent branches: pairs clearly inside or outside
    // rlist are decided from the wrapped positions; the rare band pairs (every
    // pair when the box is too small) take PD's arithmetic behind one
    // wave-uniform branch, and so do the bond-order lookups.  The pairs this lane
    // may list: a real j atom against the real i atoms, and inside the cluster
    // itself only i < j.
    const unsigned cand = (have && ob >= 0) ? (i_valid & (cj == ci ? (1u << jj) - 1u : 0xFFu)) : 0u;
    unsigned in_bits = 0, und_bits = 0;
#pragma unroll
    for (int ii = 0; ii < kClusterSize; ii++) {
      const SlotList li = s_i[wave][ii];
      const double dx = jx - li.wx, dy = jy - li.wy, dz = jz - li.wz;
      // a classification only: the band around rlist^2 (1e-10 relative) is far
      // wider than what fused multiply-adds change
      const double r2 = __builtin_fma(dx, dx, __builtin_fma(dy, dy, dz * dz));
      in_bits |= r2 < A.rlist2_lo ? 1u << ii : 0u;
      und_bits |= r2 <= A.rlist2_hi ? 1u << ii : 0u;
    }
    unsigned amb;  // pairs for PD's arithmetic
    if (A.fast) {
      lm = cand & in_bits;
      amb = cand & ~in_bits & und_bits;
    } else {
      amb = cand;
    }
    if (__ballot(amb != 0u)) {
#pragma unroll 1
      for (int ii = 0; ii < kClusterSize; ii++) {
        if ((amb >> ii) & 1u) {
          const SlotList li = s_i[wave][ii];
          const int oa = li.orig;
          // PD's arithmetic: dc = p_j - p_i, while-loop wrapping (neighbourlist.cpp:383-392)
          double ex = px[ob] - px[oa], ey = py[ob] - py[oa], ez = pz[ob] - pz[oa];
          int pimg = 13;
          bool in = true;
          if (A.periodic) {
            for (int it = 0; it < 8 && ex > A.half[0]; it++) { ex -= A.L[0]; pimg -= 9; }
            for (int it = 0; it < 8 && ex < -A.half[0]; it++) { ex += A.L[0]; pimg += 9; }
            for (int it = 0; it < 8 && ey > A.half[1]; it++) { ey -= A.L[1]; pimg -= 3; }
            for (int it = 0; it < 8 && ey < -A.half[1]; it++) { ey += A.L[1]; pimg += 3; }
            for (int it = 0; it < 8 && ez > A.half[2]; it++) { ez -= A.L[2]; pimg -= 1; }
            for (int it = 0; it < 8 && ez < -A.half[2]; it++) { ez += A.L[2]; pimg += 1; }
            const int mx = pimg / 9 - 1, my = (pimg / 3) % 3 - 1, mz = pimg % 3 - 1;
            in = (mx - (wrap_digit(lj.aux, 0) - wrap_digit(li.aux, 0))) == sx &&
                 (my - (wrap_digit(lj.aux, 1) - wrap_digit(li.aux, 1))) == sy &&
                 (mz - (wrap_digit(lj.aux, 2) - wrap_digit(li.aux, 2))) == sz;
          }
          const double er2 = ex * ex + ey * ey + ez * ez;
          if (in && er2 <= A.rlist2) lm |= 1u << ii;
        }
      }
    }
    // bond-order codes: pairs less than mid apart in index or with sparse partners
    const bool maybe = lm != 0u && ((ob > i_lo - A.mid && ob < i_hi + A.mid) || ((lj.aux >> 24) & 1) || i_sparse);
    unsigned need = 0;
    if (__ballot(maybe)) {
#pragma unroll
      for (int ii = 0; ii < kClusterSize; ii++) {
        const SlotList li = s_i[wave][ii];
        const int lo_aux = li.orig < ob ? li.aux : lj.aux;
        need |= (((lm >> ii) & 1u) && (abs(li.orig - ob) < A.mid || ((lo_aux >> 24) & 1))) ? 1u << ii : 0u;
      }
    }
    if (__ballot(need != 0u)) {
#pragma unroll 1
      for (int ii = 0; ii < kClusterSize; ii++) {
        if ((need >> ii) & 1u) {
          const SlotList li = s_i[wave][ii];
          const int oa = li.orig;
          const int lo_aux = oa < ob ? li.aux : lj.aux;
          const int code = bond_code(oa, ob, (lo_aux >> 24) & 1, A.mid, band, sp_off, sp_part, sp_ord);
          codes |= (unsigned)code << (2 * ii);
        }
      }
    }
    // one entry per (j atom, image); bit 29 of the first word: the j atom has an LJ epsilon
    const unsigned rank = A.pass == 0 ? (unsigned)min(k, kGroupRanks) : (unsigned)kGroupRanks;
    const unsigned jlj = (unsigned)((lj.aux >> 25) & 1) << 29;
    if (i_uniform) {
      const bool has = lm != 0u;
      const unsigned long long bb = __ballot(has);
      const int pos = cnt + __popcll(bb & ((1ull << lane) - 1ull));
      if (has && pos < A.stride) {
        const unsigned sm = spread8(lm);
        const int limg = jimg - wimg[0];
        E[pos] = make_uint2((unsigned)sb | ((unsigned)limg << 24) | jlj, lm | ((codes & (sm | (sm << 1))) << 8) | (rank << 24));
      }
      cnt += __popcll(bb);
    } else {
      unsigned rem = lm;
      while (__ballot(rem != 0)) {
        const bool has = rem != 0;
        unsigned m = 0;
        int limg = 0;
        if (has) {
          const int l = __ffs(rem) - 1;
          int wl = wimg[0];
#pragma unroll
          for (int q = 1; q < kClusterSize; q++)
            if (q == l) wl = wimg[q];
          limg = jimg - wl;
#pragma unroll
          for (int q = 0; q < kClusterSize; q++)
            if (((rem >> q) & 1u) && wimg[q] == wl) m |= 1u << q;
          rem &= ~m;
        }
        const unsigned long long bb = __ballot(has);
        const int pos = cnt + __popcll(bb & ((1ull << lane) - 1ull));
        if (has && pos < A.stride) {
          const unsigned sm = spread8(m);
          E[pos] = make_uint2((unsigned)sb | ((unsigned)limg << 24) | jlj, m | ((codes & (sm | (sm << 1))) << 8) | (rank << 24));
        }
        cnt += __popcll(bb);
      }
    }
  }
  if (lane == 0) {
    cl_entry_count[ci] = min(cnt, A.stride);
    // the group's work for the nonbonded dispatch order: rounds of 64 entries
    // (a pass adds the rounds its entries added to the cluster's)
    atomicAdd(&grp_work[g], ((min(cnt, A.stride) + 63) >> 6) - ((cnt0 + 63) >> 6));
    if (cnt > A.stride) atomicMax(&counter[1], (unsigned long long)cnt);
    if (cand_overflow) atomicMax(&counter[2], 1ull);  // the candidate table did not fit: more passes
    atomicAdd(&counter[0], (unsigned long long)(cnt - cnt0));
  }
}

}  // namespace

// ---------------------------------------------------------------------------------
void Engine::build_list(bool deferred) {
  require(have_positions, "positions not set");
  require(list_cutoff > 0.0, "no cutoff requested from the neighbour list");
  const int T = 256;
  const int nb_atoms = (n + T - 1) / T;
  // the whole rebuild (cleanSpace to the end of the pair search) as one timed span
  hipEvent_t span_a = nullptr;
  if (timer_sample("list_build")) {
    span_a = take_event();
    PDGPU_HIP(hipEventRecord(span_a, stream));
  }
  // 1. grid of columns (from the box alone when periodic)
  const double rlist = list_cutoff + padding;
  GridArgs g{};
  g.periodic = periodic ? 1 : 0;
  double ext[3];
  if (periodic) {
    for (int d = 0; d < 3; d++) {
      g.L[d] = box[d];
      ext[d] = box[d];
    }
    g.lo_x = -box[0] / 2.0;
    g.lo_y = -box[1] / 2.0;
  } else {
    DBuf<double> bb;
    bb.resize(6);
    hipLaunchKernelGGL(k_bbox, dim3(1), dim3(1024), 0, stream, n, x.p, y.p, z.p, bb.p);
    double hb[6];
    bb.download(hb, 6, stream);
    sync();
    for (int d = 0; d < 3; d++) ext[d] = std::max(hb[3 + d] - hb[d], 1e-3);
    g.lo_x = hb[0];
    g.lo_y = hb[1];
    for (int d = 0; d < 3; d++) g.L[d] = 0.0;
  }
  const double vol = ext[0] * ext[1] * ext[2];
  const double rho = std::max((double)n / vol, 1e-4);
  const double w_target = std::cbrt((double)kClusterSize / rho);
  g.ncx = std::max(1, std::min(4096, (int)(ext[0] / w_target)));
  g.ncy = std::max(1, std::min(4096, (int)(ext[1] / w_target)));
  g.w_x = ext[0] / g.ncx;
  g.w_y = ext[1] / g.ncy;
  if (!periodic) {  // make sure the top edge falls inside the last column
    g.w_x *= 1.0 + 1e-12;
    g.w_y *= 1.0 + 1e-12;
  }
  ncx = g.ncx;
  ncy = g.ncy;
  ncol = ncx * ncy;
  max_clusters = n / kClusterSize + ncol + 1;
  max_groups = ((max_clusters / kGroup + ncol + 1) + 7) / 8 * 8;

  wx.resize(n); wy.resize(n); wz.resize(n);
  atom_wrap.resize(n);
  atom_col.resize(n);
  col_count.resize(ncol); col_fill.resize(ncol); col_atom_start.resize(ncol);
  col_cl_start.resize(ncol); col_ncl.resize(ncol);
  col_atoms.resize(n);
  slot_orig.resize((size_t)max_clusters * kClusterSize);
  orig_slot.resize(n);
  n_clusters_d.resize(1);
  cl_col.resize(max_clusters);
  cl_lo.resize((size_t)max_clusters * 3);
  cl_hi.resize((size_t)max_clusters * 3);
  cl_entry_count.resize(max_clusters);
  entry_counter.resize(4);
  col_grp_start.resize(ncol);
  grp_first.resize(max_groups);
  grp_count.resize(max_groups);
  grp_work.resize(max_groups);
  n_groups_d.resize(1);
  wg_ncand.resize(max_groups);
  wg_cand.resize((size_t)max_groups * kGroupStride);
  const int nslots = max_clusters * kClusterSize;
  slot_list.resize((size_t)nslots * sizeof(SlotList));
  prepare_slots();

  // 2. cleanSpace (PeriodicBox only; InfiniteSpace::moveIntoBox is a no-op), which
  // also clears the column counts
  if (periodic && !h_mol_first.empty()) {
    int nm = (int)h_mol_first.size();
    hipLaunchKernelGGL(k_clean_space, dim3((std::max(nm, ncol) + T - 1) / T), dim3(T), 0, stream, nm, mol_first.p,
                       mol_last.p, x.p, y.p, z.p, box[0], box[1], box[2], ncol, col_count.p);
  } else {
    hipLaunchKernelGGL(k_fill_int, dim3((ncol + T - 1) / T), dim3(T), 0, stream, col_count.p, 0, ncol);
  }
  // 3. bins, scans and work groups, column sort and the slot records
  hipLaunchKernelGGL(k_bin, dim3(nb_atoms), dim3(T), 0, stream, n, g, x.p, y.p, z.p, wx.p, wy.p, wz.p,
                     atom_wrap.p, atom_col.p, col_count.p);
  hipLaunchKernelGGL(k_scan_columns, dim3(1), dim3(1024), 0, stream, ncol, col_count.p, col_atom_start.p,
                     col_cl_start.p, col_ncl.p, col_fill.p, col_grp_start.p, n_clusters_d.p, n_groups_d.p,
                     grp_first.p, grp_count.p, grp_work.p, entry_counter.p);
  hipLaunchKernelGGL(k_fill_columns, dim3(nb_atoms), dim3(T), 0, stream, n, atom_col.p, col_atom_start.p,
                     col_fill.p, col_atoms.p);
  const bool lj = have_nb && lj_e.n >= (size_t)n;
  const bool prm = have_nb && q_scaled.n >= (size_t)n;
  hipLaunchKernelGGL(k_sort_columns, dim3(ncol), dim3(256), 0, stream, ncol, col_count.p, col_atom_start.p,
                     col_cl_start.p, col_atoms.p, wx.p, wy.p, wz.p, atom_wrap.p, sp_off.p, lj ? lj_e.p : nullptr,
                     prm ? q_scaled.p : nullptr, prm ? lj_r.p : nullptr, prm_lo.p,
                     sprm.p, sprm_lo.p, slot_orig.p, orig_slot.p, cl_col.p,
                     reinterpret_cast<SlotList *>(slot_list.p), cl_lo.p, cl_hi.p);

  // 3. pair search
  SearchArgs A{};
  A.periodic = g.periodic;
  A.ncx = ncx;
  A.ncy = ncy;
  const double R = rlist + 1e-6 * std::max(1.0, rlist);
  A.Dx = (int)(R / g.w_x) + 1;
  A.Dy = (int)(R / g.w_y) + 1;
  A.lo_x = g.lo_x;
  A.lo_y = g.lo_y;
  A.w_x = g.w_x;
  A.w_y = g.w_y;
  // Unwrapped column offsets in [-D, D] visit each (column, image) at most once;
  // images beyond +-1 are skipped inside the kernel.
  for (int d = 0; d < 3; d++) {
    A.L[d] = periodic ? box[d] : 0.0;
    A.half[d] = periodic ? box[d] / 2.0 : 0.0;
  }
  A.rlist2 = rlist * rlist;  // sqr(Cutoff + Padding), neighbourlist.cpp:355
  // Wrapped positions differ from PD's by a few ulp of the box size, so their
  // r^2 is within ~1e-11 A^2 of PD's; pairs within 1e-10 rlist^2 of the limit
  // are decided by PD's arithmetic.
  A.rlist2_lo = A.rlist2 * (1.0 - 1e-10);
  A.rlist2_hi = A.rlist2 * (1.0 + 1e-10);
  A.fast = 1;
  if (periodic)  // inside rlist implies the minimum image only when rlist stays clear of half the box
    for (int d = 0; d < 3; d++)
      if (!(rlist * (1.0 + 1e-6) + 1e-6 < box[d] / 2.0)) A.fast = 0;
  A.Rbox2 = R * R;
  A.mid = mid;
  if (entry_capacity == 0) {
    // half of the atoms within rlist of an 8-atom cluster's box, with headroom
    double a = w_target;
    double V = a * a * a + 6 * a * a * R + 3 * Consts::PI * a * R * R + 4.0 / 3.0 * Consts::PI * R * R * R;
    double est = 0.5 * rho * V;
    int stride = (int)(est * 1.6) + 64;
    stride = (stride + 63) / 64 * 64;
    entry_capacity = (size_t)stride;
  }
  for (int attempt = 0;; attempt++) {
    A.stride = (int)entry_capacity;
    A.npass = list_passes;
    entries.resize((size_t)max_clusters * entry_capacity);
    if (attempt > 0) {  // the column scan cleared them for the first attempt
      PDGPU_HIP(hipMemsetAsync(entry_counter.p, 0, 3 * sizeof(unsigned long long), stream));
      hipLaunchKernelGGL(k_fill_int, dim3((max_groups + T - 1) / T), dim3(T), 0, stream, grp_work.p, 0, max_groups);
    }
    for (int pass = 0; pass < list_passes; pass++) {
      A.pass = pass;
      ScopedTimer t(*this, "pair_search");
      hipLaunchKernelGGL(k_pair_search, dim3(max_groups), dim3(64 * kGroup), 0, stream, A, n_groups_d.p,
                         grp_first.p, grp_count.p, cl_col.p, col_cl_start.p, col_ncl.p, cl_lo.p, cl_hi.p,
                         reinterpret_cast<const SlotList *>(slot_list.p), x.p, y.p, z.p, band.p, sp_off.p,
                         sp_part.p, sp_ord.p,
                         entries.p, cl_entry_count.p, wg_ncand.p, wg_cand.p, grp_work.p, entry_counter.p);
    }
    PDGPU_HIP(hipGetLastError());
    if (span_a) {
      hipEvent_t span_b = take_event();
      PDGPU_HIP(hipEventRecord(span_b, stream));
      timers["list_build"].pending.emplace_back(span_a, span_b);
      span_a = nullptr;
    }
    // [0] entries, [1] largest overflowing entry count, [2] candidate overflow, [3] clusters
    PDGPU_HIP(hipMemcpyAsync(h_list_check, entry_counter.p, 4 * sizeof(unsigned long long),
                             hipMemcpyDeviceToHost, stream));
    if (deferred) {
      PDGPU_HIP(hipEventRecord(list_event, stream));
      list_check_pending = true;
      break;
    }
    sync();
    n_clusters = (int)h_list_check[3];
    if (!grow_list_room()) break;
    if (attempt == 8) throw EngineError(PDGPU_ERR_CAPACITY, "neighbour list does not fit (too many neighbours)");
  }
  full_update_count++;
  prune_forced = true;
  size_eval_buffers();
  // the nonbonded kernel's dispatch order (equal work per XCD, heaviest groups
  // first) is computed by an extra workgroup of the next evaluation's prune
  nb_per_cap = 2 * ((max_groups + 7) / 8);
  grp_order.resize((size_t)8 * nb_per_cap);
  order_due = true;
  list_valid = true;
}

// After a pair search: false when everything fitted; otherwise makes room for the
// next attempt -- more passes when a work group's candidate table overflowed
// (each pass takes a disjoint share of the stencil), a larger entry capacity
// when a cluster's entries did -- and returns true.
bool Engine::grow_list_room() {
  const bool cand_over = h_list_check[2] != 0;
  const unsigned long long over = h_list_check[1];
  if (!cand_over && over == 0) return false;
  if (cand_over) {
    if (list_passes >= kMaxListPasses)
      throw EngineError(PDGPU_ERR_CAPACITY, "neighbour list candidate table overflow: more than " +
                                                std::to_string(kMaxListPasses) +
                                                " search passes would be needed (cutoff too large for the density)");
    list_passes *= 2;
  }
  if (over != 0) entry_capacity = std::max(entry_capacity * 2, (size_t)(over * 1.25 + 64) / 64 * 64);
  return true;
}

bool Engine::finish_list_check() {
  if (!list_check_pending) return true;
  PDGPU_HIP(hipEventSynchronize(list_event));
  list_check_pending = false;
  n_clusters = (int)h_list_check[3];
  if (!grow_list_room()) return true;
  list_valid = false;
  full_update_count--;  // the synchronous rebuild that follows counts this update
  return false;
}

}  // namespace pdgpu
