// Exclusive prefix sums over n values on the GPU, for compactions and table
// offsets.  The values come from a functor (value of element i) and go to
// one (element i, its value, the sum of the values before it), so that a
// scan reads and writes what its caller keeps and nothing else.
//
// Three launches: sums of tiles of kScanTile elements, one workgroup over
// those sums, then every tile again with its offset (the values are read
// twice, which costs less than writing and reading them).  Sums are below
// 2^32.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "lbm_internal.h"

namespace lbm {

constexpr uint32_t kScanBlock = 256, kScanItems = 8, kScanTile = kScanBlock * kScanItems;
inline uint32_t scan_tiles(uint64_t n) { return (uint32_t)((n + kScanTile - 1) / kScanTile); }

// Sum of v over the workgroup, and of the threads before this one.
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* red, uint32_t& before) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  uint32_t inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t up = __shfl_up(inc, o, 64);
    if (lane >= o) inc += up;
  }
  if (lane == 63) red[wv] = inc;
  __syncthreads();
  uint32_t base = 0, total = 0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
    if (w < wv) base += red[w];
    total += red[w];
  }
  before = base + inc - v;
  __syncthreads();
  return total;
}

template <class In>
__global__ void __launch_bounds__(kScanBlock)
    k_scan_sums(In in, uint32_t n, uint32_t* __restrict__ sums) {
  __shared__ uint32_t red[kScanBlock / 64];
  const uint32_t i0 = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  uint32_t v = 0;
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) v += i0 + k < n ? in(i0 + k) : 0u;
  uint32_t before;
  const uint32_t total = block_scan(v, red, before);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// sums of tiles -> sums of the tiles before; *total: all of them
static __global__ void __launch_bounds__(1024)
    k_scan_top(uint32_t* __restrict__ sums, uint32_t ntiles, uint32_t* __restrict__ total) {
  __shared__ uint32_t red[16];
  uint32_t base = 0;
  for (uint32_t t0 = 0; t0 < ntiles; t0 += 1024) {
    const uint32_t t = t0 + threadIdx.x;
    const uint32_t v = t < ntiles ? sums[t] : 0u;
    uint32_t before;
    const uint32_t all = block_scan(v, red, before);
    if (t < ntiles) sums[t] = base + before;
    base += all;
  }
  if (threadIdx.x == 0) *total = base;
}

template <class In, class Out>
__global__ void __launch_bounds__(kScanBlock)
    k_scan_write(In in, uint32_t n, const uint32_t* __restrict__ sums, Out out) {
  __shared__ uint32_t red[kScanBlock / 64];
  const uint32_t i0 = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  uint32_t v[kScanItems], sum = 0;
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    v[k] = i0 + k < n ? in(i0 + k) : 0u;
    sum += v[k];
  }
  uint32_t before;
  block_scan(sum, red, before);
  before += sums[blockIdx.x];
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    if (i0 + k < n) out(i0 + k, v[k], before);
    before += v[k];
  }
}

// The first two launches: sums (scan_tiles(n) of them) and *total.
template <class In>
int launch_scan_sums(In in, uint32_t n, uint32_t* sums, uint32_t* total, hipStream_t s) {
  const uint32_t nt = scan_tiles(n);
  if (nt) hipLaunchKernelGGL((k_scan_sums<In>), dim3(nt), dim3(kScanBlock), 0, s, in, n, sums);
  hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, s, sums, nt, total);
  LBM_HIP(hipGetLastError());
  return LBM_OK;
}

// The third.
template <class In, class Out>
int launch_scan_write(In in, uint32_t n, const uint32_t* sums, Out out, hipStream_t s) {
  const uint32_t nt = scan_tiles(n);
  if (nt)
    hipLaunchKernelGGL((k_scan_write<In, Out>), dim3(nt), dim3(kScanBlock), 0, s, in, n, sums, out);
  LBM_HIP(hipGetLastError());
  return LBM_OK;
}

// Several arrays in one device allocation: add() them, alloc(), then at().
struct DevArena {
  char* base = nullptr;
  size_t bytes = 0;
  DevArena() = default;
  DevArena(const DevArena&) = delete;
  DevArena& operator=(const DevArena&) = delete;
  ~DevArena() {
    if (base) (void)hipFree(base);
  }
  size_t add(size_t n) {
    const size_t at = bytes;
    bytes += (n + 255) / 256 * 256;
    return at;
  }
  int alloc(const char* what) {
    const hipError_t e = hipMalloc((void**)&base, bytes ? bytes : 1);
    if (e == hipSuccess) return LBM_OK;
    base = nullptr;
    return hip_fail(e, what);
  }
  template <class T>
  T* at(size_t offset) const {
    return (T*)(base + offset);
  }
};

}  // namespace lbm
