// Device pieces of the Krylov kernels: the CG's state and VectorOps' dot order (vector_ops.cpp:19-64):
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
    // every read issued ahead of the 64 dependent adds
    double v[kLanes];
#pragma unroll
    for (int j = 0; j < kLanes; ++j) v[j] = row[j];
#pragma unroll
    for (int j = 0; j < kLanes; ++j) t += v[j];
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

// The dot of a staged chunk x.y (LDS, kChunk entries of which len count) by one wave, in
// VectorOps' order.
template <typename T>
__device__ __forceinline__ double wave_staged_dot(const T* x, const T* y, int len, int l, double* row) {
  double s = 0.0;
  for (int k0 = 0; k0 < len; k0 += 16 * kLanes) {
    T xv[16], yv[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      xv[j] = x[k0 + l + j * kLanes];
      yv[j] = y[k0 + l + j * kLanes];
    }
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (k0 + l + j * kLanes < len) s += as_double(xv[j]) * as_double(yv[j]);
  }
  return lane_order_sum(s, l, len < kLanes ? len : kLanes, row);
}

// The CG's scalars on the device. A field is written by one kernel of an iteration only and read
// by the others: update_dot_kernel writes it and rz, the kernel that forms the direction
// (cg_decide) rz_next, beta and the stop's fields, so that every workgroup of a kernel derives
// the same step from the same values.
struct CgState {
  double rz, rz_next, beta, tol, rhs_norm, init_res, final_res;
  int32_t it, done, converged, indefinite, max_it, zeros;
};

// The host's copy of a solve's progress, in pinned memory: the kernel that takes the stop test after
// an iteration writes `it` (direction_kernel, or the next iteration's tiles where they form the
// direction) and, last of all, `done`, so the host neither copies nor synchronises to poll.
struct CgMirror {
  double rhs_norm, init_res, final_res;
  int32_t it, converged, indefinite, zeros, done, pad;
};

__device__ inline void mirror_stop(CgMirror* m, const CgState* st, double final_res, int it, int converged) {
  if (!m) return;
  m->rhs_norm = st->rhs_norm;
  m->init_res = st->init_res;
  m->final_res = final_res;
  m->converged = converged;
  m->indefinite = st->indefinite;
  m->zeros = st->zeros;
  __hip_atomic_store(&m->it, it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&m->done, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// What every workgroup of the kernel that forms the direction decides from the totals of r.r and r.z
// (cg.cpp:60-68): false once the solve stops, else the direction is z + beta p (it > 0) or z. The
// kernel's first thread (first) records it.
__device__ inline bool cg_decide(CgState* st, CgMirror* mirror, int it, int max_it, double tol, double rz, double rr,
                                 double rz_next, bool first, double& beta) {
  beta = 0.0;
  if (it == 0) return true;  // cg_start_kernel has decided
  const double rn = sqrt(rr);
  const bool converged = rn <= tol, stop = converged || it >= max_it;
  beta = rz_next / rz;
  if (first) {
    st->final_res = rn;
    st->rz_next = rz_next;
    st->beta = beta;
    if (converged) st->converged = 1;
    if (stop) {
      st->done = 1;
      mirror_stop(mirror, st, rn, it, converged);
    } else if (mirror) {
      __hip_atomic_store(&mirror->it, it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
  return !stop;
}

// The CG vectors of a product that forms its own direction p = z + beta p_old (launch_box_cg), and
// the chunk partials of r.r and r.z (or, n = 1, their totals).
template <typename T>
struct CgDirection {
  CgState* st;
  CgMirror* mirror;
  int64_t npart;
  const double* part;
  const T *z, *p_old;
  T* p;
};

}  // namespace fx
