// bonded_dev.hpp -- the device code of FF_Bonded's terms (bonds, angles,
// torsions and impropers, FP64), shared by the bonded kernel (k_bonded.hip),
// the nonbonded kernel, whose last workgroups take the bonded terms of the
// same evaluation (k_nonbonded.hip), and the opening kernel of a GB evaluation, whose
// first ones do (k_gb.hip).  Included by those three files only.
#pragma once

#include "engine.hpp"

namespace pdgpu {
namespace {

struct ForceSink {
  long long *fx, *fy, *fz;
  long long *lds;  // 3 x kBondedWindow accumulators, or null
  int lo;          // first atom of the window
  __device__ __forceinline__ void add3(int i, double gx, double gy, double gz) const {
    if (lds) {
      unsigned long long *l = reinterpret_cast<unsigned long long *>(lds) + (i - lo);
      atomicAdd(l, (unsigned long long)fix_from_double(gx));
      atomicAdd(l + kBondedWindow, (unsigned long long)fix_from_double(gy));
      atomicAdd(l + 2 * kBondedWindow, (unsigned long long)fix_from_double(gz));
    } else {
      fix_add(&fx[i], fix_from_double(gx));
      fix_add(&fy[i], fix_from_double(gy));
      fix_add(&fz[i], fix_from_double(gz));
    }
  }
};

// The block's four energy sums in a fixed tree order; s holds 4 x 256 doubles
// of LDS.  out receives the 4 values.
__device__ __forceinline__ void block_partial(double v0, double v1, double v2, double v3, double *s, double *out) {
  s[0 * 256 + threadIdx.x] = v0;
  s[1 * 256 + threadIdx.x] = v1;
  s[2 * 256 + threadIdx.x] = v2;
  s[3 * 256 + threadIdx.x] = v3;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int d = 0; d < 4; d++) s[d * 256 + threadIdx.x] += s[d * 256 + threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 4) out[threadIdx.x] = s[threadIdx.x * 256];
}

constexpr int kBondedThreads = 256;

// One block of 256 terms (block index blk of the bonded grid; blocks never mix
// bonds, angles and torsions), run by a whole workgroup of 256 threads.  acc:
// 3 x kBondedWindow long longs of LDS (also the 4 x 256 doubles of the energy
// tree, after the forces are flushed).  eterm (optional): the energy of each
// term, for batches that reduce it per system.
__device__ __forceinline__ void bonded_block(
    int blk, int nb, const int *__restrict__ bi, const int *__restrict__ bj, const double *__restrict__ bl,
    const double *__restrict__ bk, int na, const int *__restrict__ ai, const int *__restrict__ aa,
    const int *__restrict__ aj, const double *__restrict__ at0, const double *__restrict__ ak, int nt,
    const int *__restrict__ ti, const int *__restrict__ ta, const int *__restrict__ tb,
    const int *__restrict__ tj, const int *__restrict__ tterms, const double *__restrict__ tvn,
    const double *__restrict__ tnn, const double *__restrict__ tgamma, const double *__restrict__ x,
    const double *__restrict__ y, const double *__restrict__ z, long long *__restrict__ fx,
    long long *__restrict__ fy, long long *__restrict__ fz, double *__restrict__ partial,
    double *__restrict__ eterm, const int2 *__restrict__ win, long long *acc) {
  // block -> kind and term: bonds, then angles, then torsions, each padded to whole blocks
  const int gb = (nb + 255) / 256, ga = (na + 255) / 256;
  int t;
  if (blk < gb) {
    t = blk * 256 + (int)threadIdx.x;
    if (t >= nb) t = nb + na + nt;  // idle thread
  } else if (blk < gb + ga) {
    t = (blk - gb) * 256 + (int)threadIdx.x;
    t = t < na ? nb + t : nb + na + nt;
  } else {
    t = (blk - gb - ga) * 256 + (int)threadIdx.x;
    t = t < nt ? nb + na + t : nb + na + nt;
  }
  const int2 w = win[blk];
  const ForceSink F{fx, fy, fz, w.y > 0 ? acc : nullptr, w.x};
  if (w.y > 0) {
    for (int k = threadIdx.x; k < 3 * w.y; k += kBondedThreads) acc[(k / w.y) * kBondedWindow + k % w.y] = 0;
    __syncthreads();
  }
  double eb = 0.0, ea = 0.0, et = 0.0, vir = 0.0;
  if (t < nb) {
    const int i = bi[t], j = bj[t];
    const double k = bk[t];
    double vx = x[i] - x[j], vy = y[i] - y[j], vz = z[i] - z[j];
    const double d = sqrt(vx * vx + vy * vy + vz * vz);
    const double fm = 2 * k * (d - bl[t]);
    vir = d * fm;
    eb = k * (d - bl[t]) * (d - bl[t]);
    const double s = fm / d;
    vx *= s;
    vy *= s;
    vz *= s;
    F.add3(i, -vx, -vy, -vz);
    F.add3(j, vx, vy, vz);
  } else if (t < nb + na) {
    const int q = t - nb;
    const double k = ak[q];
    if (k != 0.0) {
      const int i = ai[q], a = aa[q], j = aj[q];
      const double ivx = x[i] - x[a], ivy = y[i] - y[a], ivz = z[i] - z[a];
      const double inv_iv = 1 / sqrt(ivx * ivx + ivy * ivy + ivz * ivz);
      const double uix = ivx * inv_iv, uiy = ivy * inv_iv, uiz = ivz * inv_iv;
      const double jvx = x[j] - x[a], jvy = y[j] - y[a], jvz = z[j] - z[a];
      const double inv_jv = 1 / sqrt(jvx * jvx + jvy * jvy + jvz * jvz);
      const double ujx = jvx * inv_jv, ujy = jvy * inv_jv, ujz = jvz * inv_jv;
      const double cs = uix * ujx + uiy * ujy + uiz * ujz;
      const double th = acos(cs);
      const double sn = sin(th);
      ea = k * (th - at0[q]) * (th - at0[q]);
      const double fm = 2 * k * (th - at0[q]);
      double bx = fm * inv_iv * (uix * cs - ujx) / sn;
      double by = fm * inv_iv * (uiy * cs - ujy) / sn;
      double bz = fm * inv_iv * (uiz * cs - ujz) / sn;
      F.add3(i, -bx, -by, -bz);
      double ax = bx, ay = by, az = bz;
      bx = fm * inv_jv * (ujx * cs - uix) / sn;
      by = fm * inv_jv * (ujy * cs - uiy) / sn;
      bz = fm * inv_jv * (ujz * cs - uiz) / sn;
      F.add3(j, -bx, -by, -bz);
      F.add3(a, ax + bx, ay + by, az + bz);
    }
  } else if (t < nb + na + nt) {
    const int q = t - nb - na;
    const int i0 = ti[q], i1 = ta[q], i2 = tb[q], i3 = tj[q];
    const double v1x = x[i0] - x[i1], v1y = y[i0] - y[i1], v1z = z[i0] - z[i1];
    const double v2x = x[i1] - x[i2], v2y = y[i1] - y[i2], v2z = z[i1] - z[i2];
    const double v3x = x[i2] - x[i3], v3y = y[i2] - y[i3], v3z = z[i2] - z[i3];
    double n1x = v1y * v2z - v1z * v2y, n1y = v1z * v2x - v1x * v2z, n1z = v1x * v2y - v1y * v2x;
    double n2x = v2y * v3z - v2z * v3y, n2y = v2z * v3x - v2x * v3z, n2z = v2x * v3y - v2y * v3x;
    double n3x = v2y * n1z - v2z * n1y, n3y = v2z * n1x - v2x * n1z, n3z = v2x * n1y - v2y * n1x;
    const double in1 = 1.0 / sqrt(n1x * n1x + n1y * n1y + n1z * n1z);
    const double in2 = 1.0 / sqrt(n2x * n2x + n2y * n2y + n2z * n2z);
    const double in3 = 1.0 / sqrt(n3x * n3x + n3y * n3y + n3z * n3z);
    const double cp = (n1x * n2x + n1y * n2y + n1z * n2z) * in1 * in2;
    const double sp = (n3x * n2x + n3y * n2y + n3z * n2z) * in3 * in2;
    n2x *= in2;
    n2y *= in2;
    n2z *= in2;
    const double phi = -atan2(sp, cp);
    const bool use_cos = fabs(sp) > 0.1;
    double c1x = 0, c1y = 0, c1z = 0, c2x = 0, c2y = 0, c2z = 0;
    if (use_cos) {
      n1x *= in1;
      n1y *= in1;
      n1z *= in1;
      c1x = in1 * (n1x * cp - n2x);
      c1y = in1 * (n1y * cp - n2y);
      c1z = in1 * (n1z * cp - n2z);
      c2x = in2 * (n2x * cp - n1x);
      c2y = in2 * (n2y * cp - n1y);
      c2z = in2 * (n2z * cp - n1z);
    } else {
      n3x *= in3;
      n3y *= in3;
      n3z *= in3;
      c1x = in3 * (n3x * sp - n2x);  // dsin/dnrml3
      c1y = in3 * (n3y * sp - n2y);
      c1z = in3 * (n3z * sp - n2z);
      c2x = in2 * (n2x * sp - n3x);  // dsin/dnrml2
      c2y = in2 * (n2y * sp - n3y);
      c2z = in2 * (n2z * sp - n3z);
    }
    double fix = 0, fiy = 0, fiz = 0, fabx = 0, faby = 0, fabz = 0, fjx = 0, fjy = 0, fjz = 0;
    const int nterms = tterms[q];
    for (int h = 0; h < nterms && h < 4; h++) {
      const double kk = tvn[4 * q + h], nn = tnn[4 * q + h], g = tgamma[4 * q + h];
      double ep, dEdphi;
      if (nn > 0) {
        ep = kk * (1.0 + cos(nn * phi + g));
        dEdphi = -nn * kk * sin(nn * phi + g);
      } else {
        double diff = phi - g;
        const double PI = 3.14159265358979323846;
        if (diff < -PI)
          diff += 2.0 * PI;
        else if (diff > PI)
          diff -= 2.0 * PI;
        ep = kk * diff * diff;
        dEdphi = 2.0 * kk * diff;
      }
      et += ep;
      if (use_cos) {
        dEdphi /= sp;
        fix += dEdphi * (v2y * c1z - v2z * c1y);
        fiy += dEdphi * (v2z * c1x - v2x * c1z);
        fiz += dEdphi * (v2x * c1y - v2y * c1x);
        fjx += dEdphi * (v2z * c2y - v2y * c2z);
        fjy += dEdphi * (v2x * c2z - v2z * c2x);
        fjz += dEdphi * (v2y * c2x - v2x * c2y);
        fabx += dEdphi * (v1z * c1y - v1y * c1z + v3y * c2z - v3z * c2y);
        faby += dEdphi * (v1x * c1z - v1z * c1x + v3z * c2x - v3x * c2z);
        fabz += dEdphi * (v1y * c1x - v1x * c1y + v3x * c2y - v3y * c2x);
      } else {
        dEdphi /= -cp;
        fix += dEdphi * ((v2y * v2y + v2z * v2z) * c1x - v2x * v2y * c1y - v2x * v2z * c1z);
        fiy += dEdphi * ((v2z * v2z + v2x * v2x) * c1y - v2y * v2z * c1z - v2y * v2x * c1x);
        fiz += dEdphi * ((v2x * v2x + v2y * v2y) * c1z - v2z * v2x * c1x - v2z * v2y * c1y);
        fjx += dEdphi * (c2y * v2z - c2z * v2y);
        fjy += dEdphi * (c2z * v2x - c2x * v2z);
        fjz += dEdphi * (c2x * v2y - c2y * v2x);
        fabx += dEdphi * (-(v2y * v1y + v2z * v1z) * c1x + (2.0 * v2x * v1y - v1x * v2y) * c1y +
                          (2.0 * v2x * v1z - v1x * v2z) * c1z + c2z * v3y - c2y * v3z);
        faby += dEdphi * (-(v2z * v1z + v2x * v1x) * c1y + (2.0 * v2y * v1z - v1y * v2z) * c1z +
                          (2.0 * v2y * v1x - v1y * v2x) * c1x + c2x * v3z - c2z * v3x);
        fabz += dEdphi * (-(v2x * v1x + v2y * v1y) * c1z + (2.0 * v2z * v1x - v1z * v2x) * c1x +
                          (2.0 * v2z * v1y - v1z * v2y) * c1y + c2y * v3x - c2x * v3y);
      }
    }
    F.add3(i0, fix, fiy, fiz);
    F.add3(i1, fabx - fix, faby - fiy, fabz - fiz);
    F.add3(i2, fjx - fabx, fjy - faby, fjz - fabz);
    F.add3(i3, -fjx, -fjy, -fjz);
  }
  if (eterm && t < nb + na + nt) eterm[t] = eb + ea + et;
  __syncthreads();  // every LDS add before the flush
  if (w.y > 0) {
    for (int k = threadIdx.x; k < 3 * w.y; k += kBondedThreads) {
      const int c = k / w.y, a = k % w.y;
      const long long v = acc[c * kBondedWindow + a];
      if (v != 0) fix_add(&(c == 0 ? fx : (c == 1 ? fy : fz))[w.x + a], v);
    }
  }
  __syncthreads();  // the flush has read acc: its space holds the energy tree now
  block_partial(eb, ea, et, vir, reinterpret_cast<double *>(acc), partial + 4 * blk);
}


__device__ __forceinline__ void bonded_block(int blk, const BondedArrays &B, const double *x, const double *y,
                                             const double *z, long long *fx, long long *fy, long long *fz,
                                             double *partial, double *eterm, long long *acc) {
  bonded_block(blk, B.nb, B.bi, B.bj, B.bl, B.bk, B.na, B.ai, B.aa, B.aj, B.at0, B.ak, B.nt, B.ti, B.ta, B.tb, B.tj,
               B.tterms, B.tvn, B.tnn, B.tgamma, x, y, z, fx, fy, fz, partial, eterm, B.win, acc);
}

}  // namespace
}  // namespace pdgpu
