// k_integrate.hip -- force/energy collection and the device-resident MD loop.
//
// The integrators restate MolecularDynamics in FP64 and PD units (m/s, J/m, kg, s):
//   velocity Verlet as PD implements it (md.cpp:805-855): v += F dt/2m, kinetic
//   energy, then v += dv; r += dt (v + dv) / A; v += dv with the same old force;
//   Langevin (md.cpp:923-1059) with PD's c0/c1/c2 coefficients and correlated
//   position/velocity noise, drawing its unit normals from Philox4x32-10.
// Expressions keep PD's evaluation order with FMA contraction off, so given the
// same forces a step reproduces the oracle's FP64 arithmetic.
#include "engine.hpp"

#include <algorithm>
#include <cmath>

namespace pdgpu {

namespace {

// The energy sums of a step in their own launch (the last step of pdgpu_md, and
// every evaluation outside it).
__global__ __launch_bounds__(kSumThreads) void k_sums(SumList L) { sum_lists(L); }

// An integrator thread's loads by slot, issued together after the loads of the
// atom's own values: the nonbonded force accumulators of its slot and, for the
// next step's opening work, its position at the last prune.  f = the total
// force in J/m (as total_force gives it).
__device__ __forceinline__ void slot_loads(int i, long long a0, long long a1, long long a2,
                                           const long long *__restrict__ nbx, const long long *__restrict__ nby,
                                           const long long *__restrict__ nbz, const int *__restrict__ orig_slot,
                                           const OpenNext &O, double conv, double f[3], int &s, SlotPos &r) {
  if (nbx != nullptr || (O.on && O.spos)) s = orig_slot[i];
  long long b0 = 0, b1 = 0, b2 = 0;
  if (nbx != nullptr) {
    b0 = nbx[s];
    b1 = nby[s];
    b2 = nbz[s];
  }
  if (O.on && O.spos) r = O.pref[s];
  f[0] = (double)(a0 + b0) * conv;
  f[1] = (double)(a1 + b1) * conv;
  f[2] = (double)(a2 + b2) * conv;
}

// Total force of atom i in J/m: the original-order accumulator plus the
// nonbonded slot-order accumulator of the atom's slot.
__device__ __forceinline__ void total_force(int i, const long long *__restrict__ fbx,
                                            const long long *__restrict__ fby, const long long *__restrict__ fbz,
                                            const long long *__restrict__ nbx, const long long *__restrict__ nby,
                                            const long long *__restrict__ nbz, const int *__restrict__ orig_slot,
                                            double conv, double &f0, double &f1, double &f2) {
  long long a = fbx[i], b = fby[i], c = fbz[i];
  if (nbx) {
    int s = orig_slot[i];
    a += nbx[s];
    b += nby[s];
    c += nbz[s];
  }
  f0 = (double)a * conv;
  f1 = (double)b * conv;
  f2 = (double)c * conv;
}


// MolecularDynamics::applyForces_BeemanIntegration (md.cpp:858-919), Thermostat
// and Barostat off.  The velocity is finished with 2 F(t)/6m at the start of a
// step (not on the protocol's first step) and the kinetic energy is taken; then
// (not on its last step) the position advances by t (v + (4 F(t) - F_old) t/6m)
// and the velocity by (5 F(t) - F_old) t/6m, and F(t) becomes the old force.
__global__ __launch_bounds__(256) void k_beeman(
    int n, double t, double conv, int first_kick, int move, const double *__restrict__ mass,
    const long long *__restrict__ fbx, const long long *__restrict__ fby, const long long *__restrict__ fbz,
    const long long *__restrict__ nbx, const long long *__restrict__ nby, const long long *__restrict__ nbz,
    const int *__restrict__ orig_slot, double *__restrict__ x, double *__restrict__ y, double *__restrict__ z,
    double *__restrict__ vx, double *__restrict__ vy, double *__restrict__ vz, double *__restrict__ fox,
    double *__restrict__ foy, double *__restrict__ foz, double *__restrict__ ke_partial, OpenNext O) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double ke = 0.0;
  double px = 0.0, py = 0.0, pz = 0.0;
  int s = 0;
  SlotPos r{};
  if (i < n) {
    // Every load of the atom's own values first, then the loads by its slot
    // (the nonbonded forces, the position at the last prune): two memory trips
    // before the arithmetic, where loads behind the branches below waited for
    // the ones before them.
    const long long a0 = fbx[i], a1 = fby[i], a2 = fbz[i];
    const double m = mass[i];
    double v[3] = {vx[i], vy[i], vz[i]};
    double fo[3] = {0.0, 0.0, 0.0}, xo[3] = {0.0, 0.0, 0.0};
    if (move) {
      fo[0] = fox[i];
      fo[1] = foy[i];
      fo[2] = foz[i];
      xo[0] = x[i];
      xo[1] = y[i];
      xo[2] = z[i];
    }
    double f[3];
    slot_loads(i, a0, a1, a2, nbx, nby, nbz, orig_slot, O, conv, f, s, r);
    const double tinvmass = t / (6.0 * m);  // t div 6m
    if (first_kick)
      for (int d = 0; d < 3; d++) v[d] += ((2.0) * f[d]) * tinvmass;
    const double mag = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);  // calcKineticEnergy, md.cpp:530
    ke = 0.5 * m * (mag * mag);
    if (move) {
      const double ia = 1 / Consts::Angstrom;
      double dr[3], dv[3];
      for (int d = 0; d < 3; d++) {
        dr[d] = t * (v[d] + (4.0 * f[d] - fo[d]) * tinvmass);
        dr[d] *= ia;
        dv[d] = (5.0 * f[d] - fo[d]) * tinvmass;
      }
      px = xo[0] + dr[0];
      py = xo[1] + dr[1];
      pz = xo[2] + dr[2];
      x[i] = px;
      y[i] = py;
      z[i] = pz;
      for (int d = 0; d < 3; d++) v[d] += dv[d];
      fox[i] = f[0];
      foy[i] = f[1];
      foz[i] = f[2];
    }
    vx[i] = v[0];
    vy[i] = v[1];
    vz[i] = v[2];
  }
  if (O.on) open_next_at(O, i, n, s, r, px, py, pz);
  block_sum4_dev(ke, ke_partial);
}

__global__ __launch_bounds__(256) void k_velocity_verlet(
    int n, double t, double conv, const double *__restrict__ mass, const long long *__restrict__ fbx,
    const long long *__restrict__ fby, const long long *__restrict__ fbz, const long long *__restrict__ nbx,
    const long long *__restrict__ nby, const long long *__restrict__ nbz, const int *__restrict__ orig_slot,
    double *__restrict__ x, double *__restrict__ y, double *__restrict__ z, double *__restrict__ vx,
    double *__restrict__ vy, double *__restrict__ vz, double *__restrict__ ke_partial, OpenNext O) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double ke = 0.0;
  double px = 0.0, py = 0.0, pz = 0.0;
  int s = 0;
  SlotPos r{};
  if (i < n) {
    // the atom's own values, then the loads by its slot (two memory trips)
    const long long a0 = fbx[i], a1 = fby[i], a2 = fbz[i];
    const double m = mass[i];
    double v0 = vx[i], v1 = vy[i], v2 = vz[i];
    const double x0 = x[i], x1 = y[i], x2 = z[i];
    double f[3];
    slot_loads(i, a0, a1, a2, nbx, nby, nbz, orig_slot, O, conv, f, s, r);
    const double f0 = f[0], f1 = f[1], f2 = f[2];
    const double tinvmass = 0.5 * t / m;
    v0 += f0 * tinvmass;  // first loop, md.cpp:820-829
    v1 += f1 * tinvmass;
    v2 += f2 * tinvmass;
    const double mag = sqrt(v0 * v0 + v1 * v1 + v2 * v2);  // calcKineticEnergy, md.cpp:530
    ke = 0.5 * m * (mag * mag);
    const double ia = 1 / Consts::Angstrom;
    const double d0 = f0 * tinvmass, d1 = f1 * tinvmass, d2 = f2 * tinvmass;  // second loop, md.cpp:838-853
    v0 += d0;
    v1 += d1;
    v2 += d2;
    double r0 = t * (v0 + d0), r1 = t * (v1 + d1), r2 = t * (v2 + d2);
    r0 *= ia;
    r1 *= ia;
    r2 *= ia;
    px = x0 + r0;
    py = x1 + r1;
    pz = x2 + r2;
    x[i] = px;
    y[i] = py;
    z[i] = pz;
    vx[i] = v0 + d0;
    vy[i] = v1 + d1;
    vz[i] = v2 + d2;
  }
  if (O.on) open_next_at(O, i, n, s, r, px, py, pz);
  block_sum4_dev(ke, ke_partial);
}


// Six unit normals per atom and step, in the order of PD's three nrand calls
// (md.cpp:1011-1013): n1x n2y | n2x n1z | n1y n2z, each pair from Box-Muller
// in the form of maths.h:155-169.
__device__ void langevin_noise(uint32_t k0, uint32_t k1, uint32_t stream, uint32_t step, uint32_t atom,
                               double out[6]) {
#pragma clang fp contract(off)
  const double TwoPI = 2.0 * Consts::PI;
  for (int k = 0; k < 3; k++) {
    uint32_t c[4] = {atom, step, stream, (uint32_t)k};
    philox_round10(c, k0, k1);
    const double u1 = uniform53(c[0], c[1]), u2 = uniform53(c[2], c[3]);
    const double l = sqrt(-2.0 * log(u1));
    out[2 * k] = l * cos((-TwoPI) * u2);
    out[2 * k + 1] = l * sin((-TwoPI) * u2);
  }
}

// ---- thermostats (md.cpp:579-660) and momentum removal (md.cpp:263-272, 412-517) ----
// With a thermostat, velocity Verlet and Beeman run as two kernels around one
// reduction (which the second one does itself, without the barostat): the velocity kick and the kinetic energy (calcKineticEnergy),
// then applyThermostat on the velocities and the moving half of the step.
struct ThermoArgs {
  int kind;          // PDGPU_NO_THERMOSTAT / PDGPU_ANDERSEN / PDGPU_BERENDSEN
  double temp, dt, tau;
  int intrate;       // Andersen: (int)(10000 * AndersenRate * dt 1e15 / N^(2/3))
  uint32_t k0, k1, stream, step;
  int baro;          // Berendsen barostat (md.cpp:677-684)
  double vol_m3;     // PeriodicBox::volume() * 1e-30
  double compress, ptarget, ptau;
  double kj;                     // kcal/mol -> J per molecule
  const double *vir_nb, *vir_b;  // InternalVirial slots (kcal/mol) of the step; null when off
};

template <int INTEG>  // PDGPU_VELOCITY_VERLET or PDGPU_BEEMAN
__global__ __launch_bounds__(256) void k_kick(int n, double t, double conv, int first_kick,
                                              const double *__restrict__ mass, const long long *__restrict__ fbx,
                                              const long long *__restrict__ fby, const long long *__restrict__ fbz,
                                              const long long *__restrict__ nbx, const long long *__restrict__ nby,
                                              const long long *__restrict__ nbz, const int *__restrict__ orig_slot,
                                              double *__restrict__ vx, double *__restrict__ vy,
                                              double *__restrict__ vz, double *__restrict__ ke_partial) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double ke = 0.0;
  if (i < n) {
    double f[3];
    total_force(i, fbx, fby, fbz, nbx, nby, nbz, orig_slot, conv, f[0], f[1], f[2]);
    const double m = mass[i];
    double v[3] = {vx[i], vy[i], vz[i]};
    if (INTEG == PDGPU_VELOCITY_VERLET) {
      const double tinvmass = 0.5 * t / m;
      for (int d = 0; d < 3; d++) v[d] += f[d] * tinvmass;
    } else if (first_kick) {
      const double tinvmass = t / (6.0 * m);
      for (int d = 0; d < 3; d++) v[d] += ((2.0) * f[d]) * tinvmass;
    }
    const double mag = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    ke = 0.5 * m * (mag * mag);
    vx[i] = v[0];
    vy[i] = v[1];
    vz[i] = v[2];
  }
  block_sum4_dev(ke, ke_partial);
}

__device__ __forceinline__ double berendsen_chi(const ThermoArgs &A, int natoms, double ekin) {
  const double Edes = 3.0 * natoms * Consts::kB * A.temp / 2.0;
  return A.kind == PDGPU_BERENDSEN ? sqrt(1.0 + A.dt * (Edes / ekin - 1.0) / A.tau) : 1.0;
}

// The kinetic energy of the step (one workgroup) and Berendsen's factor
// chi = sqrt(1 + dt (Edes/ekin - 1) / tau), Edes = 3 N kB T / 2 (md.cpp:601-617).
// With the barostat: the pressure of calcKineticEnergy, P = (2 ekin - W) / (3 V)
// in Bar (md.cpp:537-552), and applyBerendsenBarostat's scaling factor
// (1 + dt Compress (P - TargetPressure) / tau_P)^(1/3) (md.cpp:677-684).
// chi[0] = thermostat factor, chi[1] = position/box scaling, chi[2] = P (Bar).
__global__ __launch_bounds__(1024) void k_thermo_sum(const double *__restrict__ part, int count, int natoms,
                                                     ThermoArgs A, double *__restrict__ ke_slot,
                                                     double *__restrict__ chi) {
  __shared__ double s[16];
  double a = 0.0;
  for (int i = threadIdx.x; i < count; i += 1024) a += part[4 * i];
  a = wave_sum(a);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x == 0) {
    double ekin = 0.0;
    for (int k = 0; k < 16; k++) ekin += s[k];
    ke_slot[0] = ekin;
    ke_slot[1] = ke_slot[2] = ke_slot[3] = 0.0;
    chi[0] = berendsen_chi(A, natoms, ekin);
    chi[1] = 1.0;
    if (A.baro) {
      double vir = 0.0;
      if (A.vir_nb) vir += A.vir_nb[0] * A.kj;
      if (A.vir_b) vir += A.vir_b[0] * A.kj;
      const double press = (2.0 * ekin - vir) / (3.0 * A.vol_m3) / Consts::Bar2Pa;
      chi[1] = pow(1.0 + (A.dt * A.compress * (press - A.ptarget) / (A.ptau)), 1.0 / 3.0);
      chi[2] = press;
    }
  }
}

// The four draws that stand in for PD's rand() of atom `atom`: the test value
// (rand() % 10000) and uniforms in (0,1] for the two nrand calls.
__device__ void andersen_draws(uint32_t k0, uint32_t k1, uint32_t stream, uint32_t step, uint32_t atom,
                               uint32_t &test, double z[4]) {
  uint32_t a[4] = {atom, step, stream, 0x414E0000u}, b[4] = {atom, step, stream, 0x414E0001u},
           c[4] = {atom, step, stream, 0x414E0002u};
  philox_round10(a, k0, k1);
  philox_round10(b, k0, k1);
  philox_round10(c, k0, k1);
  test = a[0] % 10000u;
  z[0] = uniform53(a[2], a[3]);
  z[1] = uniform53(b[0], b[1]);
  z[2] = uniform53(b[2], b[3]);
  z[3] = uniform53(c[0], c[1]);
}

// k_thermo_sum's kinetic energy by a workgroup of 256, in every thread: each stands
// for four of the 1024 threads, so the additions and their order are the same.
__device__ __forceinline__ double thermo_ekin(const double *__restrict__ part, int count) {
  __shared__ double s[16];
  for (int q = 0; q < 4; q++) {
    double a = 0.0;
    for (int i = 256 * q + (int)threadIdx.x; i < count; i += 1024) a += part[4 * i];
    a = wave_sum(a);
    if ((threadIdx.x & 63) == 0) s[4 * q + (threadIdx.x >> 6)] = a;
  }
  __syncthreads();
  double ekin = 0.0;
  for (int k = 0; k < 16; k++) ekin += s[k];
  return ekin;
}

// With `part` (no barostat) every workgroup sums the `count` kinetic-energy partials
// itself, where a launch of one workgroup between the two kernels took 4 us and two
// gaps; the O fields make it the next step's opening kernel as well.  An NVT step of
// 12,288 atoms: 57.6 us with three kernels and k_begin_nb, 54.7 now.
template <int INTEG>
__global__ __launch_bounds__(256) void k_thermo_move(
    int n, double t, double conv, int move, ThermoArgs A, const double *__restrict__ chi,
    const double *__restrict__ part, int count, double *__restrict__ ke_slot, OpenNext O,
    const double *__restrict__ mass, const long long *__restrict__ fbx, const long long *__restrict__ fby,
    const long long *__restrict__ fbz, const long long *__restrict__ nbx, const long long *__restrict__ nby,
    const long long *__restrict__ nbz, const int *__restrict__ orig_slot, double *__restrict__ x,
    double *__restrict__ y, double *__restrict__ z, double *__restrict__ vx, double *__restrict__ vy,
    double *__restrict__ vz, double *__restrict__ fox, double *__restrict__ foy, double *__restrict__ foz) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double px = 0.0, py = 0.0, pz = 0.0;
  int s = 0;
  SlotPos r{};
  double ekin = 0.0;
  if (part) {  // uniform
    ekin = thermo_ekin(part, count);
    if (i < 4) ke_slot[i] = i == 0 ? ekin : 0.0;
  }
  if (i < n) {
    const double m = mass[i];
    double v[3] = {vx[i], vy[i], vz[i]};
    if (A.kind == PDGPU_BERENDSEN) {
      const double c = part ? berendsen_chi(A, n, ekin) : chi[0];
      for (int d = 0; d < 3; d++) v[d] *= c;
    } else if (A.kind == PDGPU_ANDERSEN) {  // applyAndersonThermostat, md.cpp:620-660
      uint32_t test;
      double zz[4];
      andersen_draws(A.k0, A.k1, A.stream, A.step, (uint32_t)i, test, zz);
      if (!((int)test > A.intrate)) {
        const double TwoPI = 2.0 * Consts::PI;
        const double sigma = sqrt(Consts::kB * A.temp / m);
        double l = sqrt(-2.0 * log(zz[0]));
        const double nx = l * cos((-TwoPI) * zz[1]) * sigma;
        l = sqrt(-2.0 * log(zz[2]));
        const double ny = l * cos((-TwoPI) * zz[3]) * sigma;  // nrand(vy, vz) draws vy again
        const double nz = l * sin((-TwoPI) * zz[3]) * sigma;
        if (!(fabs(nx) > (sigma * 4)) && !(fabs(ny) > (sigma * 4)) && !(fabs(nz) > (sigma * 4))) {
          v[0] = nx;
          v[1] = ny;
          v[2] = nz;
        }
      }
    }
    double f[3];
    slot_loads(i, fbx[i], fby[i], fbz[i], nbx, nby, nbz, orig_slot, O, conv, f, s, r);
    const double ia = 1 / Consts::Angstrom;
    if (A.baro) {  // WorkSpace::scaleSystem (workspace.cpp:362-369), before the move
      const double fac = chi[1];
      x[i] *= fac;
      y[i] *= fac;
      z[i] *= fac;
    }
    if (INTEG == PDGPU_VELOCITY_VERLET) {  // second loop, md.cpp:836-854
      const double tinvmass = 0.5 * t / m;
      double dr[3];
      for (int d = 0; d < 3; d++) {
        const double dv = f[d] * tinvmass;
        v[d] += dv;
        dr[d] = t * (v[d] + dv);
        dr[d] *= ia;
        v[d] += dv;
      }
      x[i] += dr[0];
      y[i] += dr[1];
      z[i] += dr[2];
    } else if (move) {  // Beeman, md.cpp:894-918
      const double tinvmass = t / (6.0 * m);
      const double fo[3] = {fox[i], foy[i], foz[i]};
      double dr[3], dv[3];
      for (int d = 0; d < 3; d++) {
        dr[d] = t * (v[d] + (4.0 * f[d] - fo[d]) * tinvmass);
        dr[d] *= ia;
        dv[d] = (5.0 * f[d] - fo[d]) * tinvmass;
      }
      x[i] += dr[0];
      y[i] += dr[1];
      z[i] += dr[2];
      for (int d = 0; d < 3; d++) v[d] += dv[d];
      fox[i] = f[0];
      foy[i] = f[1];
      foz[i] = f[2];
    }
    vx[i] = v[0];
    vy[i] = v[1];
    vz[i] = v[2];
    px = x[i];
    py = y[i];
    pz = z[i];
  }
  if (O.on) open_next_at(O, i, n, s, r, px, py, pz);
}

// Sums for the momentum step: mass, m v, m p, m (p x v) (p in A), 10 per block.
__global__ __launch_bounds__(256) void k_mom_partials(int n, const double *__restrict__ mass,
                                                      const double *__restrict__ x, const double *__restrict__ y,
                                                      const double *__restrict__ z, const double *__restrict__ vx,
                                                      const double *__restrict__ vy, const double *__restrict__ vz,
                                                      double *__restrict__ part) {
  __shared__ double s[4][10];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double a[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (i < n) {
    const double m = mass[i], p[3] = {x[i], y[i], z[i]}, v[3] = {vx[i], vy[i], vz[i]};
    a[0] = m;
    for (int d = 0; d < 3; d++) {
      a[1 + d] = v[d] * m;
      a[4 + d] = p[d] * m;
    }
    a[7] = (p[1] * v[2] - p[2] * v[1]) * m;
    a[8] = (p[2] * v[0] - p[0] * v[2]) * m;
    a[9] = (p[0] * v[1] - p[1] * v[0]) * m;
  }
  for (int k = 0; k < 10; k++) a[k] = wave_sum(a[k]);
  if ((threadIdx.x & 63) == 0)
    for (int k = 0; k < 10; k++) s[threadIdx.x >> 6][k] = a[k];
  __syncthreads();
  if (threadIdx.x < 10) part[10 * blockIdx.x + threadIdx.x] = s[0][threadIdx.x] + s[1][threadIdx.x] +
                                                                s[2][threadIdx.x] + s[3][threadIdx.x];
}

// One workgroup: mom = linear momentum (3), angular momentum (3), centre of mass
// (3, A), |L|.  L = A (sum m p x v - com x P), the sum of md.cpp:466-475.
__global__ __launch_bounds__(256) void k_mom_finish(const double *__restrict__ part, int count,
                                                    double *__restrict__ mom) {
  __shared__ double s[4][10];
  double a[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int b = threadIdx.x; b < count; b += 256)
    for (int k = 0; k < 10; k++) a[k] += part[10 * b + k];
  for (int k = 0; k < 10; k++) a[k] = wave_sum(a[k]);
  if ((threadIdx.x & 63) == 0)
    for (int k = 0; k < 10; k++) s[threadIdx.x >> 6][k] = a[k];
  __syncthreads();
  if (threadIdx.x == 0) {
    double t[10];
    for (int k = 0; k < 10; k++) t[k] = s[0][k] + s[1][k] + s[2][k] + s[3][k];
    const double M = t[0], P[3] = {t[1], t[2], t[3]};
    const double com[3] = {t[4] / M, t[5] / M, t[6] / M};
    double L[3];
    L[0] = (t[7] - (com[1] * P[2] - com[2] * P[1])) * Consts::Angstrom;
    L[1] = (t[8] - (com[2] * P[0] - com[0] * P[2])) * Consts::Angstrom;
    L[2] = (t[9] - (com[0] * P[1] - com[1] * P[0])) * Consts::Angstrom;
    for (int d = 0; d < 3; d++) {
      mom[d] = P[d];
      mom[3 + d] = L[d];
      mom[6 + d] = com[d];
    }
    mom[9] = sqrt(L[0] * L[0] + L[1] * L[1] + L[2] * L[2]);
  }
}

// zeroTotalLinearMomentum then zeroTotalAngularMomentum (md.cpp:480-517), both
// dividing by (iend - istart) = N - 1.
__global__ __launch_bounds__(256) void k_mom_apply(int n, const double *__restrict__ mass,
                                                   const double *__restrict__ x, const double *__restrict__ y,
                                                   const double *__restrict__ z, double *__restrict__ vx,
                                                   double *__restrict__ vy, double *__restrict__ vz,
                                                   const double *__restrict__ mom) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double m = mass[i], nm1 = (double)(n - 1);
  double v[3] = {vx[i], vy[i], vz[i]};
  for (int d = 0; d < 3; d++) v[d] -= mom[d] / (nm1 * m);
  const double L[3] = {mom[3], mom[4], mom[5]};
  const double p[3] = {(x[i] - mom[6]) * Consts::Angstrom, (y[i] - mom[7]) * Consts::Angstrom,
                       (z[i] - mom[8]) * Consts::Angstrom};
  double t[3] = {L[1] * p[2] - L[2] * p[1], L[2] * p[0] - L[0] * p[2], L[0] * p[1] - L[1] * p[0]};
  const double tm = sqrt(t[0] * t[0] + t[1] * t[1] + t[2] * t[2]);
  if (tm != 0)
    for (int d = 0; d < 3; d++) t[d] /= tm;
  const double pm = sqrt(p[0] * p[0] + p[1] * p[1] + p[2] * p[2]);
  for (int d = 0; d < 3; d++) {
    t[d] *= mom[9] / pm;
    t[d] /= nm1 * m;
    v[d] -= t[d];
  }
  vx[i] = v[0];
  vy[i] = v[1];
  vz[i] = v[2];
}

struct LangevinArgs {
  double t, gamma, gammat, temp;
  double c0, c1, c2, varr, varv, crv;
  int first_kick;   // Step > 0
  int move;         // Step < Steps-1
  uint32_t k0, k1, stream, step;
  double conv;
  // 0: the whole step in one kernel; with a barostat two kernels around the
  // pressure reduction: 1 = kick + kinetic energy, 2 = scaling (scale[1]) + move
  int phase;
  const double *scale;
};

__global__ __launch_bounds__(256) void k_langevin(
    int n, LangevinArgs L, const double *__restrict__ mass, const long long *__restrict__ fbx,
    const long long *__restrict__ fby, const long long *__restrict__ fbz, const long long *__restrict__ nbx,
    const long long *__restrict__ nby, const long long *__restrict__ nbz, const int *__restrict__ orig_slot,
    double *__restrict__ x, double *__restrict__ y, double *__restrict__ z, double *__restrict__ vx,
    double *__restrict__ vy, double *__restrict__ vz, double *__restrict__ ke_partial, OpenNext O) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double ke = 0.0;
  double px = 0.0, py = 0.0, pz = 0.0;
  int si = 0;
  SlotPos ri{};
  if (i < n) {
    // the atom's own values, then the loads by its slot (two memory trips)
    const long long a0 = fbx[i], a1 = fby[i], a2 = fbz[i];
    const double m = mass[i];
    double v[3] = {vx[i], vy[i], vz[i]};
    double xo[3] = {x[i], y[i], z[i]};
    double f[3];
    slot_loads(i, a0, a1, a2, nbx, nby, nbz, orig_slot, O, L.conv, f, si, ri);
    const double t = L.t;
    const double tinvmass = t / m;
    if (L.first_kick && L.phase != 2) {
      for (int d = 0; d < 3; d++) v[d] += (1.0 - L.c0 / L.c1) * f[d] * tinvmass / L.gammat;
    }
    const double mag = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    ke = 0.5 * m * (mag * mag);
    if (L.phase == 2) {  // applyBarostat between the kick and the move (md.cpp:1022-1023)
      const double fac = L.scale[1];
      for (int d = 0; d < 3; d++) xo[d] *= fac;
    }
    if (L.move && L.phase != 1) {
      const double kTdivm = Consts::kB * L.temp / m;
      const double sigmav = sqrt(kTdivm * L.varv);
      const double sigmar = sqrt(kTdivm * L.varr) / L.gamma;
      double z6[6];
      langevin_noise(L.k0, L.k1, L.stream, L.step, (uint32_t)i, z6);
      const double n1[3] = {z6[0], z6[4], z6[3]};  // n1x n1y n1z
      const double n2[3] = {z6[2], z6[1], z6[5]};  // n2x n2y n2z
      const double s = sqrt(1.0 - L.crv * L.crv);
      const double ia = 1 / Consts::Angstrom;
      double dr[3], dv[3];
      for (int d = 0; d < 3; d++) {
        const double delv = sigmav * (L.crv * n1[d] + s * n2[d]);
        const double delr = sigmar * n1[d];
        dr[d] = t * (L.c1 * v[d] + L.c2 * f[d] * tinvmass) + delr;
        dr[d] *= ia;
        dv[d] = (L.c0 * L.c2) * f[d] * tinvmass / L.c1 + delv;
      }
      for (int d = 0; d < 3; d++) xo[d] += dr[d];
      for (int d = 0; d < 3; d++) {
        v[d] *= L.c0;
        v[d] += dv[d];
      }
    }
    if (L.phase == 2 || (L.move && L.phase != 1)) {
      x[i] = xo[0];
      y[i] = xo[1];
      z[i] = xo[2];
    }
    vx[i] = v[0];
    vy[i] = v[1];
    vz[i] = v[2];
    px = xo[0];
    py = xo[1];
    pz = xo[2];
  }
  if (O.on) open_next_at(O, i, n, si, ri, px, py, pz);
  if (L.phase != 2) block_sum4_dev(ke, ke_partial);  // uniform over the grid
}

}  // namespace

void Engine::flush_sums(const StepRecord *rec) {
  if (pending_sums.empty() && !rec) return;
  size_t k = 0;
  do {  // more than kMaxSums entries: several launches, in order
    SumList L{};
    for (; k < pending_sums.size() && L.n < kMaxSums; k++, L.n++) {
      L.part[L.n] = pending_sums[k].part;
      L.out[L.n] = pending_sums[k].out;
      L.count[L.n] = pending_sums[k].count;
    }
    const bool last = k == pending_sums.size();
    L.record = (last && rec) ? 1 : 0;
    if (rec) L.rec = *rec;
    L.e_out = e_out.p;
    hipLaunchKernelGGL(k_sums, dim3(1), dim3(kSumThreads), 0, stream, L);
  } while (k < pending_sums.size());
  pending_sums.clear();
  PDGPU_HIP(hipGetLastError());
}

// The sums of an MD step wait for a workgroup of the next step's nonbonded or GB opening
// kernel, which saves a launch per step; more lists than one workgroup takes run now.
void Engine::defer_step_sums(const StepRecord &rec) {
  if (pending_sums.size() > (size_t)kMaxSums) {
    flush_sums(&rec);
    return;
  }
  SumList L{};
  for (size_t k = 0; k < pending_sums.size(); k++, L.n++) {
    L.part[L.n] = pending_sums[k].part;
    L.out[L.n] = pending_sums[k].out;
    L.count[L.n] = pending_sums[k].count;
  }
  L.record = 1;
  L.rec = rec;
  L.e_out = e_out.p;
  pending_sums.clear();
  fused_sums = L;
  fused_pending = true;
}

// e_out layout (doubles): [0..3] nonbonded vdw, elec, virial, -; [4..7] bonded
// bond, angle, torsion, virial; [8..11] GB pol, vdw, elec, virial (see k_gb.hip);
// [12] GB self; [13..16] LCPO cavity energy (slot 13); [20] kinetic energy (J); others spare.
void Engine::run_fused_sums() {
  hipLaunchKernelGGL(k_sums, dim3(1), dim3(kSumThreads), 0, stream, fused_sums);
  PDGPU_HIP(hipGetLastError());
  fused_pending = false;
}

void Engine::evaluate(uint32_t components, int step, bool flush) {
  const bool eonly = (components & PDGPU_ENERGY_ONLY) != 0;
  const bool nbon = (components & PDGPU_NONBONDED) != 0;
  pending_sums.clear();
  if (flush) fused_pending = false;  // only pdgpu_md's steps hand their sums on
  const bool gbon = (components & PDGPU_GB) != 0, tiled = gbon && have_gb && !gb->plain;
  const bool opened = !flush && opened_ahead && (nbon ? list_valid : tiled);
  opened_ahead = false;
  if (nbon && !list_valid) build_list();
  begin_evaluation(nbon, nullptr, opened, tiled);
  const bool bon = (components & PDGPU_BONDED) && (nbonds + nangles + ntors) > 0;
  if (nbon) launch_nonbonded(e_out.p + 0, !eonly, nullptr, bon ? e_out.p + 4 : nullptr);
  const bool gb_bonded = bon && !nbon && tiled;
  if (bon && !nbon && !gb_bonded) launch_bonded(e_out.p + 4);
  // the GB sums share the launch of the surface energies
  const bool share = tiled && (components & PDGPU_SASA) && !eonly;
  if (gbon) launch_gb(e_out.p + 8, eonly, gb_bonded ? e_out.p + 4 : nullptr, !share);
  const GBSums G = share ? gb->sum_args(e_out.p, 8, 8) : GBSums{};
  if (components & PDGPU_SASA) launch_lcpo(e_out.p + 13, step, step < 0, eonly, share ? &G : nullptr);
  last_components = components;
  if (flush) flush_sums();
}

namespace {
// The total force of atoms first .. first + n - 1 in PD's units (J/m), AoS: the fixed-point sums of
// the bonded / GB / LCPO accumulators and of the atom's nonbonded slot, converted
// on the device so that one array of doubles crosses to the host.
__global__ void k_forces_jm(int first, int n, double conv, const long long *__restrict__ fbx, const long long *__restrict__ fby,
                            const long long *__restrict__ fbz, const long long *__restrict__ nbx,
                            const long long *__restrict__ nby, const long long *__restrict__ nbz,
                            const int *__restrict__ orig_slot, double *__restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x, i = first + k;
  if (k >= n) return;
  long long fx = fbx[i], fy = fby[i], fz = fbz[i];
  if (nbx) {
    const int s = orig_slot[i];
    fx += nbx[s];
    fy += nby[s];
    fz += nbz[s];
  }
  out[3 * k] = __dmul_rn((double)fx, conv);
  out[3 * k + 1] = __dmul_rn((double)fy, conv);
  out[3 * k + 2] = __dmul_rn((double)fz, conv);
}
}  // namespace

void Engine::forces_to_host(double *f, size_t stride_bytes) {
  const bool nbon = (last_components & PDGPU_NONBONDED) != 0;
  const double conv = Consts::kcalA_to_Jm() / kFixScale;
  // the kernel stores to pinned host memory, in pieces for large systems
  double *h = stage.need((size_t)3 * std::min(n, kStagePiece));
  for (int first = 0; first < n; first += kStagePiece) {
    const int m = std::min(kStagePiece, n - first);
    hipLaunchKernelGGL(k_forces_jm, dim3((m + 255) / 256), dim3(256), 0, stream, first, m, conv, fbx.p, fby.p, fbz.p,
                       nbon ? nbx.p : nullptr, nby.p, nbz.p, orig_slot.p, h);
    PDGPU_HIP(hipGetLastError());
    sync();
    // PD's contract: the component adds into wspace.cur.atom[i].f
    char *at = reinterpret_cast<char *>(f) + (size_t)first * stride_bytes;
    for (int i = 0; i < m; i++) {
      double *p = reinterpret_cast<double *>(at + (size_t)i * stride_bytes);
      p[0] += h[3 * i];
      p[1] += h[3 * i + 1];
      p[2] += h[3 * i + 2];
    }
  }
}

void Engine::energies_to_host(uint32_t components, pdgpu_energies *out) {
  e_out.download(h_eout, 24, stream);
  sync();
  energies_from_slots(components, h_eout, out);
}

// The energy slots (kcal/mol, layout of evaluate) as PD's Hamiltonian terms in J.
void Engine::energies_from_slots(uint32_t components, const double *h, pdgpu_energies *out) const {
  const double kj = Consts::kcal_to_J();
  pdgpu_energies e{};
  if (components & PDGPU_NONBONDED) {
    const double cor = nbk.vdwcor_per_atom * n;
    e.epot_vdw += (h[0] + cor) * kj;
    e.epot_elec += h[1] * kj;
    e.virial += h[2] * kj;
    e.epot += (h[0] + h[1] + cor) * kj;
  }
  if (components & PDGPU_BONDED) {
    e.epot_bond += h[4] * kj;
    e.epot_angle += h[5] * kj;
    e.epot_torsion += h[6] * kj;
    e.virial += h[7] * kj;
    e.epot += (h[4] + h[5] + h[6]) * kj;
  }
  if (components & PDGPU_GB)
    gb_slots_to_energies(h + 8, gb->prm.FastMode != 0 || (components & PDGPU_ENERGY_ONLY) != 0, e);
  if (components & PDGPU_SASA) {
    e.epot_surf += h[13] * kj;
    e.epot += h[13] * kj;
  }
  *out = e;
}

void Engine::integrate(const pdgpu_md_params &p, int step, double *ke_slot, bool open) {
  const int T = 256;
  const int grid = (n + T - 1) / T;
  e_partial_ke.resize((size_t)grid * 4);
  OpenNext O{};
  open = open && p.barostat == PDGPU_NO_BAROSTAT && (last_components & (PDGPU_NONBONDED | PDGPU_GB)) && step < p.total_steps - 1;
  if (open && !(last_components & PDGPU_NONBONDED)) {
    O.on = 1;
    O.fbx = fbx.p;
    O.fby = fby.p;
    O.fbz = fbz.p;
    opened_ahead = true;
  } else if (open) {
    O = OpenNext{1, dmax_cur ^ 1, spos.p, spos32.p, pref.p, prune_dmax.p, nbx.p, nby.p, nbz.p, fbx.p, fby.p, fbz.p};
    opened_ahead = true;
  }
  const bool nbon = (last_components & PDGPU_NONBONDED) != 0;
  const long long *ax = nbon ? nbx.p : nullptr, *ay = nbon ? nby.p : nullptr, *az = nbon ? nbz.p : nullptr;
  const double conv = Consts::kcalA_to_Jm() / kFixScale;
  const double gammat = p.fric_coeff * p.timestep;
  const bool beeman = p.integrator == PDGPU_BEEMAN;
  // Langevin with gamma*dt < 1e-5 falls back to velocity Verlet (md.cpp:966-971)
  const bool vv = !beeman && (p.integrator == PDGPU_VELOCITY_VERLET || gammat < 0.00001);
  if (beeman && fox.n < (size_t)n) {  // the workspace's old forces start at zero
    fox.resize(n);
    foy.resize(n);
    foz.resize(n);
    PDGPU_HIP(hipMemsetAsync(fox.p, 0, n * sizeof(double), stream));
    PDGPU_HIP(hipMemsetAsync(foy.p, 0, n * sizeof(double), stream));
    PDGPU_HIP(hipMemsetAsync(foz.p, 0, n * sizeof(double), stream));
  }
  const bool baro = p.barostat == PDGPU_BERENDSEN_BAROSTAT;
  ThermoArgs A{};
  if (baro) {
    require(periodic, "the Berendsen barostat needs a PeriodicBox (its pressure needs a volume)");
    require(p.pressure_tau > 0 && p.compress > 0, "BerendsenPressureTau and Compress must be positive");
    // the step's virial sums are needed now, not with the next step's first kernel
    flush_sums();
    A.baro = 1;
    A.vol_m3 = box[0] * box[1] * box[2] * 1E-30;
    A.compress = p.compress;
    A.ptarget = p.target_pressure;
    A.ptau = p.pressure_tau;
    A.kj = Consts::kcal_to_J();
    A.vir_nb = (last_components & PDGPU_NONBONDED) ? e_out.p + 2 : nullptr;
    A.vir_b = ((last_components & PDGPU_BONDED) && (nbonds + nangles + ntors) > 0) ? e_out.p + 7 : nullptr;
    A.dt = p.timestep;
    thermo.resize(4);
  } else {
    require(p.barostat == PDGPU_NO_BAROSTAT, "unknown barostat");
  }
  if ((beeman || vv) && (p.thermostat != PDGPU_NO_THERMOSTAT || baro)) {
    // kick + kinetic energy, applyThermostat and applyBarostat, then the moving
    // half (md.cpp:831-834, 890-892)
    A.kind = p.thermostat;
    A.temp = p.temperature;
    A.dt = p.timestep;
    A.tau = p.berendsen_tau;
    const double rate = p.andersen_rate * p.timestep * 1E15 / std::pow(double(n), double(2.0 / 3.0));
    A.intrate = (int)(10000.0 * rate);
    A.k0 = (uint32_t)p.seed;
    A.k1 = (uint32_t)(p.seed >> 32);
    A.stream = p.noise_stream;
    A.step = (uint32_t)step;
    thermo.resize(4);
    const int first = step > 0 ? 1 : 0, move = step < (p.total_steps - 1) ? 1 : 0;
    if (beeman)
      hipLaunchKernelGGL(k_kick<PDGPU_BEEMAN>, dim3(grid), dim3(T), 0, stream, n, p.timestep, conv, first, mass.p,
                         fbx.p, fby.p, fbz.p, ax, ay, az, orig_slot.p, vx.p, vy.p, vz.p, e_partial_ke.p);
    else
      hipLaunchKernelGGL(k_kick<PDGPU_VELOCITY_VERLET>, dim3(grid), dim3(T), 0, stream, n, p.timestep, conv, first,
                         mass.p, fbx.p, fby.p, fbz.p, ax, ay, az, orig_slot.p, vx.p, vy.p, vz.p, e_partial_ke.p);
    // every workgroup reads all partials, so their traffic grows with the square of the
    // atoms; past 131,072 the sum keeps its own launch, and the barostat needs its factor
    // on the host
    const bool own_sum = baro || grid > 512;
    const double *part = own_sum ? nullptr : e_partial_ke.p;
    if (own_sum)
      hipLaunchKernelGGL(k_thermo_sum, dim3(1), dim3(1024), 0, stream, e_partial_ke.p, grid, n, A, ke_slot, thermo.p);
    if (beeman)
      hipLaunchKernelGGL(k_thermo_move<PDGPU_BEEMAN>, dim3(grid), dim3(T), 0, stream, n, p.timestep, conv, move, A,
                         thermo.p, part, grid, ke_slot, O, mass.p, fbx.p, fby.p, fbz.p, ax, ay, az, orig_slot.p, x.p,
                         y.p, z.p, vx.p, vy.p, vz.p, fox.p, foy.p, foz.p);
    else
      hipLaunchKernelGGL(k_thermo_move<PDGPU_VELOCITY_VERLET>, dim3(grid), dim3(T), 0, stream, n, p.timestep, conv,
                         move, A, thermo.p, part, grid, ke_slot, O, mass.p, fbx.p, fby.p, fbz.p, ax, ay, az, orig_slot.p, x.p, y.p, z.p,
                         vx.p, vy.p, vz.p, nullptr, nullptr, nullptr);
    PDGPU_HIP(hipGetLastError());
    return;
  }
  if (beeman) {
    hipLaunchKernelGGL(k_beeman, dim3(grid), dim3(T), 0, stream, n, p.timestep, conv, step > 0 ? 1 : 0,
                       step < (p.total_steps - 1) ? 1 : 0, mass.p, fbx.p, fby.p, fbz.p, ax, ay, az, orig_slot.p,
                       x.p, y.p, z.p, vx.p, vy.p, vz.p, fox.p, foy.p, foz.p, e_partial_ke.p, O);
  } else if (vv) {
    hipLaunchKernelGGL(k_velocity_verlet, dim3(grid), dim3(T), 0, stream, n, p.timestep, conv, mass.p, fbx.p,
                       fby.p, fbz.p, ax, ay, az, orig_slot.p, x.p, y.p, z.p, vx.p, vy.p, vz.p, e_partial_ke.p, O);
  } else {
    LangevinArgs L{};
    L.t = p.timestep;
    L.gamma = p.fric_coeff;
    L.gammat = gammat;
    L.temp = p.temperature;
    langevin_coefficients(gammat, &L.c0);
    L.first_kick = step > 0 ? 1 : 0;
    L.move = step < (p.total_steps - 1) ? 1 : 0;
    L.k0 = (uint32_t)p.seed;
    L.k1 = (uint32_t)(p.seed >> 32);
    L.stream = p.noise_stream;
    L.step = (uint32_t)step;
    L.conv = conv;
    if (baro) {  // kick + kinetic energy, the pressure and scaling factor, then scaling + move
      A.kind = PDGPU_NO_THERMOSTAT;
      L.phase = 1;
      hipLaunchKernelGGL(k_langevin, dim3(grid), dim3(T), 0, stream, n, L, mass.p, fbx.p, fby.p, fbz.p, ax, ay,
                         az, orig_slot.p, x.p, y.p, z.p, vx.p, vy.p, vz.p, e_partial_ke.p, OpenNext{});
      hipLaunchKernelGGL(k_thermo_sum, dim3(1), dim3(1024), 0, stream, e_partial_ke.p, grid, n, A, ke_slot,
                         thermo.p);
      L.phase = 2;
      L.scale = thermo.p;
      hipLaunchKernelGGL(k_langevin, dim3(grid), dim3(T), 0, stream, n, L, mass.p, fbx.p, fby.p, fbz.p, ax, ay,
                         az, orig_slot.p, x.p, y.p, z.p, vx.p, vy.p, vz.p, nullptr, OpenNext{});
      PDGPU_HIP(hipGetLastError());
      return;
    }
    hipLaunchKernelGGL(k_langevin, dim3(grid), dim3(T), 0, stream, n, L, mass.p, fbx.p, fby.p, fbz.p, ax, ay, az,
                       orig_slot.p, x.p, y.p, z.p, vx.p, vy.p, vz.p, e_partial_ke.p, O);
  }
  PDGPU_HIP(hipGetLastError());
  defer_sum4(e_partial_ke.p, grid, ke_slot);
}

// calcTotalLinearMomentum .. zeroTotalAngularMomentum (md.cpp:263-272, 412-517).
void Engine::remove_momentum() {
  const int T = 256;
  const int grid = (n + T - 1) / T;
  mom_part.resize((size_t)grid * 10);
  mom.resize(10);
  hipLaunchKernelGGL(k_mom_partials, dim3(grid), dim3(T), 0, stream, n, mass.p, x.p, y.p, z.p, vx.p, vy.p, vz.p,
                     mom_part.p);
  hipLaunchKernelGGL(k_mom_finish, dim3(1), dim3(256), 0, stream, mom_part.p, grid, mom.p);
  hipLaunchKernelGGL(k_mom_apply, dim3(grid), dim3(T), 0, stream, n, mass.p, x.p, y.p, z.p, vx.p, vy.p, vz.p,
                     mom.p);
  PDGPU_HIP(hipGetLastError());
}

// c0 c1 c2 varr varv crv of applyForces_LangevinIntegration (md.cpp:947-986).
void langevin_coefficients(double gammat, double *c) {
  const double gt = gammat, gt2 = gt * gt, gt3 = gt * gt2, gt4 = gt2 * gt2, gt5 = gt2 * gt3, gt6 = gt3 * gt3,
               gt7 = gt3 * gt4, gt8 = gt4 * gt4, gt9 = gt4 * gt5;
  double c0, c1, c2, varr, varv, crv;
  if (gammat > 0.05) {
    c0 = std::exp(-gammat);
    c1 = (1 - c0) / gammat;
    c2 = (1 - c1) / gammat;
    const double eg = std::exp(-gammat);
    varv = (1.0 - eg * eg);
    varr = (2.0 * gammat - 3.0 + (4.0 - eg) * eg);
    crv = (1.0 - eg) * (1.0 - eg) / (std::sqrt(varv * varr));
  } else {
    c0 = 1 - gt + 0.5 * gt2 - gt3 / 6.0 + gt4 / 24.0 - gt5 / 120.0 + gt6 / 720.0 - gt7 / 5040.0 + gt8 / 40320.0 -
         gt9 / 362880.0;
    c1 = 1 - (0.5 * gt - gt2 / 6.0 + gt3 / 24.0 - gt4 / 120.0 + gt5 / 720.0 - gt6 / 5040.0 + gt7 / 40320.0 -
              gt8 / 362880.0);
    c2 = 0.5 - gt / 6.0 + gt2 / 24.0 - gt3 / 120.0 + gt4 / 720.0 - gt5 / 5040.0 + gt6 / 40320.0 - gt7 / 362880.0;
    varr = 2.0 * gt3 / 3.0 - gt4 / 2.0 + 7.0 * gt5 / 30.0 - gt6 / 12.0 + 31.0 * gt7 / 1260.0 - gt8 / 160.0 +
           127.0 * gt9 / 90720.0;
    varv = 2.0 * gt - 2.0 * gt2 + 4.0 * gt3 / 3.0 - 2.0 * gt4 / 3.0 + 4.0 * gt5 / 15.0 - 4.0 * gt6 / 45.0 +
           8.0 * gt7 / 315.0 - 2.0 * gt8 / 315.0 + 4.0 * gt9 / 2835.0;
    crv = std::sqrt(3.0) * (0.5 - 3.0 * gt / 16.0 - 17.0 * gt2 / 1280.0 + 17.0 * gt3 / 6144.0 +
                            40967.0 * gt4 / 34406400.0 - 57203.0 * gt5 / 275251200.0 -
                            1429487.0 * gt6 / 13212057600.0);
  }
  c[0] = c0;
  c[1] = c1;
  c[2] = c2;
  c[3] = varr;
  c[4] = varv;
  c[5] = crv;
}

namespace {
// A trajectory frame (ProtocolBase::UpdateTra): the positions and the step's
// energy slots into frame f of the frame buffers.
__global__ void k_copy_frame(int n, const double *__restrict__ x, const double *__restrict__ y,
                             const double *__restrict__ z, const double *__restrict__ e_out, int f,
                             double *__restrict__ fxyz, double *__restrict__ fe) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double *F = fxyz + (size_t)f * 3 * n;
  if (i < n) {
    F[i] = x[i];
    F[n + i] = y[i];
    F[2 * n + i] = z[i];
  }
  if (i < 24) fe[24 * f + i] = e_out[i];
}
}  // namespace

// MolecularDynamics::run_core (md.cpp:219-284): refresh the list every
// UpdateNList steps (protocolbase.cpp:135-144), evaluate forces, integrate.
void Engine::md(const pdgpu_md_params &p, int n_steps, double *epot_trace, double *ekin_trace) {
  require(have_positions, "positions not set");
  require(vx.n >= (size_t)n && mass.n >= (size_t)n, "velocities or masses not set");
  require(p.timestep > 0, "timestep must be positive");
  require((p.components & PDGPU_ENERGY_ONLY) == 0, "MD needs forces: PDGPU_ENERGY_ONLY is for pdgpu_compute");
  trace.resize((size_t)std::max(n_steps, 1) * 2);
  fused_pending = false;
  opened_ahead = false;
  const uint32_t comp = p.components;
  const double cor = (comp & PDGPU_NONBONDED) ? nbk.vdwcor_per_atom * n : 0.0;
  // every(Step + m_StepOffset, UpdateTra) (protocolbase.cpp:251-257): step > 0
  auto is_frame = [&](int step) { return p.update_tra > 0 && step > 0 && step % p.update_tra == 0; };
  int n_frames = 0;
  for (int s = 0; s < n_steps; s++) n_frames += is_frame(p.step_offset + s) ? 1 : 0;
  h_frame_steps.clear();
  if (n_frames > 0) {
    frame_xyz.resize((size_t)n_frames * 3 * n);
    frame_e.resize((size_t)n_frames * 24);
  }
  frame_components = comp;
  for (int s = 0; s < n_steps; s++) {
    const int step = p.step_offset + s;
    const bool rebuild = (comp & (PDGPU_NONBONDED)) && p.update_nlist > 0 && (step % p.update_nlist) == 0;
    if (rebuild) build_list(true);
    evaluate(comp, step, false);
    if (rebuild && !finish_list_check()) {  // the list overflowed: rebuild with room and evaluate again
      build_list();
      evaluate(comp, step, false);
    }
    // the integrator opens the next step's evaluation when that step keeps the
    // list and this one records no frame (whose sums run now, not deferred)
    const bool next_rebuild =
        (comp & PDGPU_NONBONDED) && p.update_nlist > 0 && ((step + 1) % p.update_nlist) == 0;
    const bool open = (comp & (PDGPU_NONBONDED | PDGPU_GB)) && s + 1 < n_steps && !next_rebuild && !is_frame(step);
    integrate(p, step, e_out.p + 20, open);
    if (p.barostat == PDGPU_BERENDSEN_BAROSTAT) {
      // PeriodicBox::scale: the box follows the positions; the next step's
      // kernels (basis vectors, list build) take the new edge lengths
      double h[4];
      thermo.download(h, 4, stream);
      sync();
      for (int d = 0; d < 3; d++) box[d] *= h[1];
      last_pressure = h[2];
    }
    // every(Step, UpdateRemoveTotalMomentum) with a thermostat (md.cpp:263-272, protocolbase.cpp:251-257)
    if (p.thermostat != PDGPU_NO_THERMOSTAT && p.remove_momentum > 0 && step > 0 && step % p.remove_momentum == 0)
      remove_momentum();
    const StepRecord rec{trace.p, s, (comp & PDGPU_NONBONDED) ? 1 : 0, (comp & PDGPU_BONDED) ? 1 : 0,
                         (comp & PDGPU_GB) ? 1 : 0, (comp & PDGPU_SASA) ? 1 : 0, cor, Consts::kcal_to_J()};
    if (is_frame(step)) {  // outtra.append(): this step's sums now, then the frame
      flush_sums(&rec);
      const int f = (int)h_frame_steps.size();
      hipLaunchKernelGGL(k_copy_frame, dim3((std::max(n, 24) + 255) / 256), dim3(256), 0, stream, n, x.p, y.p, z.p,
                         e_out.p, f, frame_xyz.p, frame_e.p);
      PDGPU_HIP(hipGetLastError());
      h_frame_steps.push_back(step);
    } else {
      defer_step_sums(rec);
    }
  }
  if (fused_pending) run_fused_sums();  // the last step's
  TraceFetch tf;
  const double *h = tf.get(stage, trace, (size_t)n_steps * 2, stream);
  bool nan = false;
  for (int s = 0; s < n_steps; s++) {
    if (epot_trace) epot_trace[s] = h[2 * s];
    if (ekin_trace) ekin_trace[s] = h[2 * s + 1];
    if (std::isnan(h[2 * s])) nan = true;
  }
  if (nan) throw EngineError(PDGPU_ERR_UNSTABLE, "Simulation unstable or division by zero");
}

}  // namespace pdgpu
