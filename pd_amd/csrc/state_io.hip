// state_io.hip -- positions and velocities between the caller's arrays and the device.
//
// PD keeps one record per atom (72 bytes apart), the device three arrays.  The
// vectors go through pinned host memory that the kernels below read or write over
// the bus, splitting or joining the components on the way: one launch and one wait
// per call, where three copies of pageable arrays took the runtime's staging three
// times.  A call moves little, so what bounds it is the count of waits: the positions
// of one of 256 small systems took 54 us and take 14, set_positions with 11
// energy-only updates of 1,536 atoms 981 -> 576 us, set_positions, list and forces of
// 98,304 atoms 845 -> 722.  Large systems go in pieces, so the pinned memory stays
// small.
#include <algorithm>
#include <cstring>

#include "engine.hpp"

namespace pdgpu {

namespace {

__global__ void k_split_xyz(int n, const double *__restrict__ src, double *__restrict__ x, double *__restrict__ y,
                            double *__restrict__ z) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  x[i] = src[3 * i];
  y[i] = src[3 * i + 1];
  z[i] = src[3 * i + 2];
}

__global__ void k_join_xyz(int n, const double *__restrict__ x, const double *__restrict__ y,
                           const double *__restrict__ z, double *__restrict__ dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  dst[3 * i] = x[i];
  dst[3 * i + 1] = y[i];
  dst[3 * i + 2] = z[i];
}

}  // namespace

void xyz_to_device(HostStage &st, hipStream_t s, const double *xyz, size_t stride_bytes, int n, double *x, double *y,
                   double *z) {
  double *h = st.need((size_t)3 * std::min(n, kStagePiece));
  const char *src = reinterpret_cast<const char *>(xyz);
  for (int a = 0; a < n; a += kStagePiece) {
    const int m = std::min(kStagePiece, n - a);
    const char *p = src + (size_t)a * stride_bytes;
    if (stride_bytes == 3 * sizeof(double))
      std::memcpy(h, p, (size_t)m * stride_bytes);
    else
      for (int i = 0; i < m; i++) std::memcpy(h + 3 * (size_t)i, p + (size_t)i * stride_bytes, 3 * sizeof(double));
    hipLaunchKernelGGL(k_split_xyz, dim3((m + 255) / 256), dim3(256), 0, s, m, h, x + a, y + a, z + a);
    PDGPU_HIP(hipGetLastError());
    PDGPU_HIP(hipStreamSynchronize(s));  // the buffer is free for the next piece or call
  }
}

void xyz_to_host(HostStage &st, hipStream_t s, const double *x, const double *y, const double *z, int n, double *xyz,
                 size_t stride_bytes) {
  double *h = st.need((size_t)3 * std::min(n, kStagePiece));
  char *dst = reinterpret_cast<char *>(xyz);
  for (int a = 0; a < n; a += kStagePiece) {
    const int m = std::min(kStagePiece, n - a);
    hipLaunchKernelGGL(k_join_xyz, dim3((m + 255) / 256), dim3(256), 0, s, m, x + a, y + a, z + a, h);
    PDGPU_HIP(hipGetLastError());
    PDGPU_HIP(hipStreamSynchronize(s));
    char *p = dst + (size_t)a * stride_bytes;
    if (stride_bytes == 3 * sizeof(double))
      std::memcpy(p, h, (size_t)m * stride_bytes);
    else
      for (int i = 0; i < m; i++) std::memcpy(p + (size_t)i * stride_bytes, h + 3 * (size_t)i, 3 * sizeof(double));
  }
}

}  // namespace pdgpu
