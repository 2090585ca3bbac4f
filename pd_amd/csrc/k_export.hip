// k_export.hip -- the neighbour list in PD's packed form, for host force fields.
//
// The list lives in cluster entries (k_list.hip).  PD's form is, per atom, the words
// j | bond order << 24 | image << 27 in ascending j (neighbourlist.h:131-151,
// neighbourlist.cpp:422).  On the device: one pass over the entries counts each
// atom's pairs, one places the words in the atoms' rows, and a workgroup per atom sorts
// its row in LDS (bitonic, on the word rotated so that j leads; j is unique in a
// row).  The rows then cross the bus in pieces of 4 MiB through pinned memory, one
// piece in flight while the caller's array takes the one before it.  Count and
// rows of 12,288 atoms (4.5 M pairs): 244 ms when the host expanded and sorted the
// entries, now 1.5 ms: half kernels (sort 149 us, fill 132, search 77), half the
// caller's 18 MB of fresh pages.
#include <algorithm>
#include <cstring>

#include "engine.hpp"

namespace pdgpu {

namespace {

constexpr int kRowMax = 8192;              // words a workgroup sorts in LDS (32 KiB); longer rows on the host
constexpr size_t kPieceWords = 1 << 20;    // 4 MiB

// An entry of the list as PD's rows see it: its own atoms ii (bits of `row_b`) go to
// the j atom's row, the j atom to theirs (bits of `row_a`).  A pair stands in the row of
// its higher index, and with the shadow list in both.
struct Entry {
  int ob;         // the j atom
  int img;        // image of p_j - p_ii
  unsigned lm;    // listed atoms of the cluster
  unsigned codes;
  unsigned row_a, row_b;
};

__device__ __forceinline__ Entry read_entry(uint2 e, const int *__restrict__ slot_orig, const int *oa, int shadow) {
  Entry r;
  r.ob = slot_orig[e.x & 0xFFFFFFu];
  r.img = (int)((e.x >> 24) & 31u);
  r.lm = e.y & 0xFFu;
  r.codes = e.y >> 8;
  unsigned higher = 0u;
#pragma unroll
  for (int ii = 0; ii < kClusterSize; ii++) higher |= (oa[ii] > r.ob ? 1u : 0u) << ii;
  r.row_a = shadow ? r.lm : r.lm & higher;
  r.row_b = shadow ? r.lm : r.lm & ~higher;
  return r;
}

// One wavefront per cluster: the listed pairs of its entries, added to *total.
__global__ __launch_bounds__(64) void k_export_total(const int *__restrict__ cl_count,
                                                     const uint2 *__restrict__ entries, size_t stride,
                                                     unsigned long long *__restrict__ total) {
  const int ci = blockIdx.x, cnt = cl_count[ci];
  int s = 0;
  for (int k = threadIdx.x; k < cnt; k += 64) s += __popc(entries[ci * stride + k].y & 0xFFu);
  for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
  if (threadIdx.x == 0 && s) atomicAdd(total, (unsigned long long)s);
}

// One atomic per entry for the j atom's row and eight per cluster for its own atoms:
// device-scope atomics bound this (one per pair and row: 244 us for 4.5 M pairs, with
// k_export_fill 328; now 25 and 132).
__global__ __launch_bounds__(64) void k_export_count(const int *__restrict__ cl_count,
                                                     const uint2 *__restrict__ entries, size_t stride,
                                                     const int *__restrict__ slot_orig, int shadow,
                                                     int *__restrict__ row_count) {
  const int ci = blockIdx.x, cnt = cl_count[ci], lane = threadIdx.x;
  int oa[kClusterSize], own = 0;
#pragma unroll
  for (int ii = 0; ii < kClusterSize; ii++) oa[ii] = slot_orig[ci * kClusterSize + ii];
  for (int k0 = 0; k0 < cnt; k0 += 64) {
    Entry e{};
    if (k0 + lane < cnt) e = read_entry(entries[ci * stride + k0 + lane], slot_orig, oa, shadow);
    if (e.row_b) atomicAdd(&row_count[e.ob], __popc(e.row_b));
#pragma unroll
    for (int ii = 0; ii < kClusterSize; ii++) {
      const int c = __popcll(__ballot((e.row_a >> ii) & 1u));
      own += lane == ii ? c : 0;
    }
  }
  if (own) atomicAdd(&row_count[slot_orig[ci * kClusterSize + lane]], own);  // lanes 0..7
}

// left: the words each row still takes (its count at the start, zero at the end)
__global__ __launch_bounds__(64) void k_export_fill(const int *__restrict__ cl_count,
                                                    const uint2 *__restrict__ entries, size_t stride,
                                                    const int *__restrict__ slot_orig, int shadow, int periodic,
                                                    const unsigned long long *__restrict__ row_start,
                                                    int *__restrict__ left, uint32_t *__restrict__ packed) {
  const int ci = blockIdx.x, cnt = cl_count[ci], lane = threadIdx.x;
  int oa[kClusterSize];
#pragma unroll
  for (int ii = 0; ii < kClusterSize; ii++) oa[ii] = slot_orig[ci * kClusterSize + ii];
  auto word = [&](int j, unsigned codes, int ii, int img) {
    const unsigned c = (codes >> (2 * ii)) & 3u;
    return (uint32_t)j | ((c == 0u ? 7u : c) << 24) | (periodic ? (uint32_t)img << 27 : 0u);
  };
  for (int k0 = 0; k0 < cnt; k0 += 64) {
    Entry e{};
    if (k0 + lane < cnt) e = read_entry(entries[ci * stride + k0 + lane], slot_orig, oa, shadow);
    if (e.row_b) {
      unsigned long long at = row_start[e.ob] + (unsigned)atomicSub(&left[e.ob], __popc(e.row_b));
#pragma unroll
      for (int ii = 0; ii < kClusterSize; ii++)
        if ((e.row_b >> ii) & 1u) packed[--at] = word(oa[ii], e.codes, ii, 26 - e.img);
    }
#pragma unroll
    for (int ii = 0; ii < kClusterSize; ii++) {
      const unsigned long long m = __ballot((e.row_a >> ii) & 1u);
      if (m == 0ull) continue;  // uniform
      int end = 0;
      if (lane == 0) end = atomicSub(&left[oa[ii]], __popcll(m));
      end = __shfl(end, 0, 64);
      if ((e.row_a >> ii) & 1u)
        packed[row_start[oa[ii]] + (unsigned)(end - 1 - __popcll(m & ((1ull << lane) - 1ull)))] =
            word(e.ob, e.codes, ii, e.img);
    }
  }
}

// A workgroup per row; dynamic LDS holds the longest row sorted here, to a power of two.
__global__ __launch_bounds__(256) void k_export_sort(const unsigned long long *__restrict__ row_start,
                                                     uint32_t *__restrict__ packed) {
  extern __shared__ uint32_t key[];
  uint32_t *row = packed + row_start[blockIdx.x];
  const int n = (int)(row_start[blockIdx.x + 1] - row_start[blockIdx.x]);
  if (n < 2 || n > kRowMax) return;  // uniform
  int size = 2;
  while (size < n) size <<= 1;
  for (int k = threadIdx.x; k < size; k += 256) {
    const uint32_t w = k < n ? row[k] : 0xFFFFFFFFu;
    key[k] = (w << 8) | (w >> 24);
  }
  for (int len = 2; len <= size; len <<= 1)
    for (int half = len >> 1; half > 0; half >>= 1) {
      __syncthreads();
      for (int t = threadIdx.x; t < size / 2; t += 256) {
        const int a = 2 * half * (t / half) + t % half, b = a + half;
        const uint32_t u = key[a], v = key[b];
        if ((u > v) == ((a & len) == 0)) {
          key[a] = v;
          key[b] = u;
        }
      }
    }
  __syncthreads();
  for (int k = threadIdx.x; k < n; k += 256) row[k] = (key[k] >> 8) | (key[k] << 24);
}

__global__ void k_export_clear(int n, int *__restrict__ a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0;
}

}  // namespace

int64_t Engine::count_pairs() {
  require(list_valid, "no neighbour list built");
  if (n_clusters == 0) return 0;
  ex_total.resize(1);
  PDGPU_HIP(hipMemsetAsync(ex_total.p, 0, sizeof(unsigned long long), stream));
  hipLaunchKernelGGL(k_export_total, dim3(n_clusters), dim3(64), 0, stream, cl_entry_count.p, entries.p,
                     (size_t)entry_capacity, ex_total.p);
  PDGPU_HIP(hipGetLastError());
  unsigned long long t = 0;
  ex_total.download(&t, 1, stream);
  sync();
  return (int64_t)t * (calc_shadow ? 2 : 1);
}

// counts: n ints; packed: room for `capacity` words.
void Engine::export_pairs(int32_t *counts, uint32_t *packed, int64_t capacity) {
  require(list_valid, "no neighbour list built");
  ex_count.resize(n);
  hipLaunchKernelGGL(k_export_clear, dim3((n + 255) / 256), dim3(256), 0, stream, n, ex_count.p);
  if (n_clusters > 0)
    hipLaunchKernelGGL(k_export_count, dim3(n_clusters), dim3(64), 0, stream, cl_entry_count.p, entries.p,
                       (size_t)entry_capacity, slot_orig.p, calc_shadow ? 1 : 0, ex_count.p);
  PDGPU_HIP(hipGetLastError());
  std::vector<int> cnt(n);
  ex_count.download(cnt.data(), n, stream);
  sync();
  std::vector<unsigned long long> start((size_t)n + 1, 0);
  int longest = 0;
  for (int i = 0; i < n; i++) {
    start[i + 1] = start[i] + (unsigned)cnt[i];
    longest = std::max(longest, std::min(cnt[i], kRowMax));
  }
  const size_t total = start[n];
  require((int64_t)total <= capacity, "capacity too small for the pair set");
  std::copy(cnt.begin(), cnt.end(), counts);
  if (total == 0) return;
  ex_start.upload(start, stream);
  ex_packed.resize(total);
  hipLaunchKernelGGL(k_export_fill, dim3(n_clusters), dim3(64), 0, stream, cl_entry_count.p, entries.p,
                     (size_t)entry_capacity, slot_orig.p, calc_shadow ? 1 : 0, periodic ? 1 : 0, ex_start.p,
                     ex_count.p, ex_packed.p);
  int size = 2;
  while (size < longest) size <<= 1;
  hipLaunchKernelGGL(k_export_sort, dim3(n), dim3(256), size * sizeof(uint32_t), stream, ex_start.p, ex_packed.p);
  PDGPU_HIP(hipGetLastError());
  // the copy of one piece runs while the caller's array takes the piece before it
  uint32_t *buf = reinterpret_cast<uint32_t *>(stage.need((std::min(total, 2 * kPieceWords) + 1) / 2));
  auto words = [&](size_t piece) { return std::min(kPieceWords, total - piece * kPieceWords); };
  const size_t pieces = (total + kPieceWords - 1) / kPieceWords;
  for (size_t p = 0; p <= pieces; p++) {
    if (p > 0) sync();  // piece p - 1 has arrived
    if (p < pieces)
      PDGPU_HIP(hipMemcpyAsync(buf + (p & 1) * kPieceWords, ex_packed.p + p * kPieceWords,
                               words(p) * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
    if (p > 0)
      std::memcpy(packed + (p - 1) * kPieceWords, buf + ((p - 1) & 1) * kPieceWords, words(p - 1) * sizeof(uint32_t));
  }
  for (int i = 0; i < n; i++)  // rows too long for LDS
    if (cnt[i] > kRowMax)
      std::sort(packed + start[i], packed + start[i + 1],
                [](uint32_t a, uint32_t b) { return (a & 0xFFFFFFu) < (b & 0xFFFFFFu); });
}

}  // namespace pdgpu
