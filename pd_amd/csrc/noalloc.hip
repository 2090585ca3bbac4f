// noalloc.hip -- pdgpu_compute_noalloc: a force/energy evaluation that allocates
// nothing, for callers that cannot allocate device memory (code under stream
// capture, tight serving loops, harnesses that forbid hipMalloc).
//
// The evaluation uses the same kernels as pdgpu_compute.  What pdgpu_compute
// keeps in engine buffers sized per call -- the per-workgroup energy partials of
// the nonbonded and bonded kernels and the reduced energy slots -- lives here in
// one file-scope device array, `scratch`, of kScratchDoubles doubles (1 MiB).
// Each GPU holds its own copy of the array until the process ends; its device
// address is looked up once per device (scratch_for_device, called when an
// engine is created on that device).  Every buffer the kernels write besides
// these was sized by the last pdgpu_build_list, and the forces go to a device
// array the caller owns.
//
// All engines on one GPU share that GPU's scratch array and it keeps the last
// call's contents: each call clears the energy slots it sums into, and writes
// every partial before reading it.  Calls on one GPU that overlap in time (two
// host threads, or two engines' streams running concurrently) race on it.
#include <mutex>

#include "engine.hpp"

namespace pdgpu {

constexpr size_t kScratchDoubles = size_t(1) << 17;  // 1 MiB
constexpr size_t kScratchSlots = 32;                 // energy slots (24 used), then the partials
static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
double *g_scratch[kMaxDevices] = {};

// f[i] += (fb[i] + nb[slot of i]) * conv in PD's AoS layout (stride in doubles);
// the product and the sum are rounded separately, as the host conversion does.
__global__ void k_forces_to_device(int n, double conv, const long long *__restrict__ fbx,
                                   const long long *__restrict__ fby, const long long *__restrict__ fbz,
                                   const long long *__restrict__ nbx, const long long *__restrict__ nby,
                                   const long long *__restrict__ nbz, const int *__restrict__ orig_slot,
                                   double *__restrict__ f, size_t stride) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  long long fx = fbx[i], fy = fby[i], fz = fbz[i];
  if (nbx) {
    const int s = orig_slot[i];
    fx += nbx[s];
    fy += nby[s];
    fz += nbz[s];
  }
  double *p = f + (size_t)i * stride;
  p[0] = __dadd_rn(p[0], __dmul_rn((double)fx, conv));
  p[1] = __dadd_rn(p[1], __dmul_rn((double)fy, conv));
  p[2] = __dadd_rn(p[2], __dmul_rn((double)fz, conv));
}

}  // namespace

double *scratch_for_device(int device) {
  if (device < 0 || device >= kMaxDevices) throw EngineError(PDGPU_ERR_ARG, "device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch[device]) {
    int cur = 0;
    PDGPU_HIP(hipGetDevice(&cur));
    PDGPU_HIP(hipSetDevice(device));
    void *ptr = nullptr;
    const hipError_t err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    (void)hipSetDevice(cur);
    if (err != hipSuccess || !ptr)
      throw EngineError(PDGPU_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(err));
    g_scratch[device] = static_cast<double *>(ptr);
  }
  return g_scratch[device];
}

void Engine::evaluate_noalloc(uint32_t components, double *d_f, size_t stride_bytes, pdgpu_energies *out) {
  const uint32_t allowed = PDGPU_NONBONDED | PDGPU_BONDED | PDGPU_ENERGY_ONLY;
  require((components & ~allowed) == 0,
          "pdgpu_compute_noalloc evaluates PDGPU_NONBONDED and PDGPU_BONDED (with or without PDGPU_ENERGY_ONLY)");
  require(components & (PDGPU_NONBONDED | PDGPU_BONDED), "no component selected");
  require(have_positions, "positions not set");
  require(!(d_f && (components & PDGPU_ENERGY_ONLY)), "PDGPU_ENERGY_ONLY computes no forces: f_accum must be NULL");
  require(!d_f || (stride_bytes >= 3 * sizeof(double) && stride_bytes % sizeof(double) == 0),
          "the force stride must be a multiple of 8 bytes and at least 24");
  require(scratch != nullptr, "scratch array not set up");
  const bool nbon = (components & PDGPU_NONBONDED) != 0;
  const bool eonly = (components & PDGPU_ENERGY_ONLY) != 0;
  const bool bon = (components & PDGPU_BONDED) && (nbonds + nangles + ntors) > 0;
  // every engine buffer the kernels write must exist already: nothing is resized here
  require(fbx.n >= (size_t)n && e_out.n >= 24, "engine buffers not sized: build the neighbour list first");
  if (nbon) {
    require(have_nb, "nonbonded component not set up");
    require(list_valid, "the neighbour list is not built (pdgpu_compute_noalloc never rebuilds it)");
    const size_t nslots = (size_t)max_clusters * kClusterSize;
    require(spos.n >= nslots && spos32.n >= nslots && pref.n >= nslots && prune_dmax.n > 0 &&
                pentries.n >= (size_t)max_clusters * entry_capacity &&
                pcount.n >= (size_t)max_clusters &&
                pcount_nolj.n >= (size_t)max_clusters,
            "engine buffers not sized: build the neighbour list first");
  }
  const size_t n_nb = nbon ? (size_t)max_groups * nb_parts * 4 : 0;
  const size_t n_b = bon ? (size_t)bonded_blocks(nbonds, nangles, ntors) * 4 : 0;
  const size_t need = kScratchSlots + n_nb + n_b;
  if (need > kScratchDoubles)
    throw EngineError(PDGPU_ERR_ARG, "system too large for pdgpu_compute_noalloc: its energy partials need " +
                                         std::to_string(need) + " doubles of scratch, the maximum is " +
                                         std::to_string(kScratchDoubles));
  double *eo = scratch;
  double *p_nb = scratch + kScratchSlots;
  double *p_b = p_nb + n_nb;
  pending_sums.clear();
  fused_pending = false;
  begin_evaluation(nbon, eo);  // clears the accumulators and the energy slots in scratch
  if (nbon) launch_nonbonded(eo + 0, !eonly, p_nb);
  if (bon) launch_bonded(eo + 4, p_b);
  last_components = components;
  flush_sums();
  if (d_f) {
    const double conv = Consts::kcalA_to_Jm() / kFixScale;
    hipLaunchKernelGGL(k_forces_to_device, dim3((n + 255) / 256), dim3(256), 0, stream, n, conv, fbx.p, fby.p,
                       fbz.p, nbon ? nbx.p : nullptr, nby.p, nbz.p, orig_slot.p, d_f, stride_bytes / sizeof(double));
    PDGPU_HIP(hipGetLastError());
  }
  PDGPU_HIP(hipMemcpyAsync(h_eout, eo, 24 * sizeof(double), hipMemcpyDeviceToHost, stream));
  sync();
  energies_from_slots(components, h_eout, out);
}

}  // namespace pdgpu

extern "C" int pdgpu_compute_noalloc(pdgpu_engine *h, uint32_t components, double *d_f_accum,
                                     size_t stride_bytes, pdgpu_energies *energies) {
  pdgpu::Engine *e = reinterpret_cast<pdgpu::Engine *>(h);
  if (!e) return PDGPU_ERR_ARG;
  try {
    PDGPU_HIP(hipSetDevice(e->device));
    pdgpu_energies tmp;
    e->evaluate_noalloc(components, d_f_accum, stride_bytes, &tmp);
    if (energies) *energies = tmp;
    if (tmp.epot != tmp.epot)
      throw pdgpu::EngineError(PDGPU_ERR_UNSTABLE, "Simulation unstable or division by zero");
    return PDGPU_OK;
  } catch (const pdgpu::EngineError &x) {
    e->last_error = x.what();
    return x.code;
  } catch (const std::exception &x) {
    e->last_error = x.what();
    return PDGPU_ERR_ARG;
  }
}
