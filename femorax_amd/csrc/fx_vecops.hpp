// Device pieces of VectorOps' dot order (vector_ops.cpp:19-64) shared by the Krylov kernels:
// chunks of 2048 entries, lane l of 64 summing entries l, l + 64, ... of its chunk, the lane sums
// added in lane order, chunk sums reduced level by level the same way.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fx {

constexpr int kChunk = 2048;
constexpr int kLanes = 64;
// A vector kernel's workgroup takes one chunk with four waves, eight entries per thread: every
// load of the chunk is in flight at once (one round of memory latency; a wave that walked its 32
// entries per lane in turn took 8 to 11 us for a chunk of a small solve, all of it latency).
constexpr int kVecThreads = 256;
constexpr int kPerThread = kChunk / kVecThreads;
// A reduction of at most this many chunk partials is done by every workgroup that needs its
// total (16 loads per lane, from L2) instead of by a launch of its own: a launch costs about 4 us
// of a small solve's iteration, while at 3,121 partials (6.4 M equations) the repeated reads of
// 3,121 workgroups would cost more than the launch saves.
constexpr int64_t kInlineParts = 1024;

__host__ __device__ inline int64_t chunks(int64_t n) { return (n + kChunk - 1) / kChunk; }

__device__ __forceinline__ double as_double(double v) { return v; }
__device__ __forceinline__ double as_double(float v) { return static_cast<double>(v); }

// The lane sums of a wave added in lane order, through a row of 64 doubles in LDS (a wave's LDS
// accesses complete in program order); the lanes past `lanes` hold 0. The total in every lane.
__device__ __forceinline__ double lane_order_sum(double s, int l, int lanes, double* row) {
  row[l] = s;
  __builtin_amdgcn_wave_barrier();
  double t = 0.0;
  if (lanes == kLanes) {
#pragma unroll 16
    for (int j = 0; j < kLanes; ++j) t += row[j];
  } else {
    for (int j = 0; j < lanes; ++j) t += row[j];
  }
  __builtin_amdgcn_wave_barrier();
  return t;
}

// sum of src[(begin + k) * stride], k < len <= 2048, by one wave: eight loads in flight per lane.
// The total in every lane. (Entries past len add 0.0, which changes no bit of a sum from 0.0.)
__device__ __forceinline__ double wave_chunk_sum(const double* src, int64_t stride, int64_t begin, int64_t len, int l,
                                                 double* row) {
  double s = 0.0;
  for (int64_t k0 = 0; k0 < len; k0 += 8 * kLanes) {
    double v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int64_t k = k0 + l + j * kLanes;
      v[j] = k < len ? src[(begin + k) * stride] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) s += v[j];
  }
  return lane_order_sum(s, l, static_cast<int>(len < kLanes ? len : kLanes), row);
}

// A total from its chunk partials (npart <= kInlineParts <= one chunk), by one wave.
__device__ __forceinline__ double wave_total(const double* part, int nv, int v, int64_t npart, int l, double* row) {
  if (npart <= 1) return part[v];
  return wave_chunk_sum(part + v, nv, 0, npart, l, row);
}

// The dot of a staged chunk x.y (LDS, entries 0..len) by one wave, in VectorOps' order.
template <typename T>
__device__ __forceinline__ double wave_staged_dot(const T* x, const T* y, int len, int l, double* row) {
  double s = 0.0;
  if (len == kChunk) {
#pragma unroll
    for (int j = 0; j < kChunk / kLanes; ++j) s += as_double(x[l + j * kLanes]) * as_double(y[l + j * kLanes]);
  } else {
    for (int k = l; k < len; k += kLanes) s += as_double(x[k]) * as_double(y[k]);
  }
  return lane_order_sum(s, l, len < kLanes ? len : kLanes, row);
}

}  // namespace fx
