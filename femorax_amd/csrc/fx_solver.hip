// Device-resident Krylov solvers for the hex8 operator.
//
// ConjugateGradient::solve with Jacobi (src/solvers/cg.cpp:24-72, jacobi.cpp:10-26) with its
// scalars kept on the device: each kernel reads a `done` flag and becomes a no-op once the
// stop rule ||r|| <= max(rtol ||b||, atol) (cg.cpp:34, 60) or p.Ap <= 0 (cg.cpp:49-53) has
// fired, so the host may queue iterations ahead of the progress the device reports
// (fx_cg_watch.hpp) and the iterate is exactly the one the reference stops at. Dot products follow VectorOps' order (vector_ops.cpp:19-64): chunks of
// 2048 entries, 64 lanes, lane l summing entries l, l+64, ...; lane sums in lane order; chunk
// sums reduced level by level. They accumulate in FP64 whatever the vector type.
//
// The mixed-precision solve wraps an FP32 CG (FP32 operator and vectors, FP64 dots) in FP64
// iterative refinement: r = b - A x with the FP64 operator, d = A32^-1 r approximately,
// x += d in FP64, until the FP64 residual meets the same stop rule.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <mutex>
#include <string>

#include "fx_cg_watch.hpp"
#include "fx_internal.hpp"
#include "fx_kernels.hpp"
#include "fx_vecops.hpp"

namespace fx {

// Partial sums per chunk of x.y in VectorOps' lane order (one workgroup per chunk, see
// kVecThreads). 27,744 entries (14 chunks): 11.2 -> 3 us; 6.4 M entries: HBM-bound either way.
template <typename T>
__global__ __launch_bounds__(kVecThreads) void chunk_dot_kernel(int64_t n, const T* __restrict__ x,
                                                                const T* __restrict__ y, double* __restrict__ partial,
                                                                const int32_t* done) {
  __shared__ T xs[kChunk], ys[kChunk];
  __shared__ double row[kLanes];
  const int stopped = done ? *done : 0;
  const int64_t begin = static_cast<int64_t>(blockIdx.x) * kChunk;
  const int len = static_cast<int>(n - begin < kChunk ? n - begin : kChunk);
  const int t = threadIdx.x;
  T xv[kPerThread], yv[kPerThread];
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    const int k = t + j * kVecThreads;
    const int64_t i = begin + (k < len ? k : 0);  // unconditional, so that all are in flight
    xv[j] = x[i];
    yv[j] = y[i];
  }
  if (stopped) return;
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    xs[t + j * kVecThreads] = xv[j];
    ys[t + j * kVecThreads] = yv[j];
  }
  __syncthreads();
  if (t >= kLanes) return;
  const double s = wave_staged_dot(xs, ys, len, t, row);
  if (t == 0) partial[blockIdx.x] = s;
}

// Reduce `nv` (1 or 2) interleaved sequences of chunk partials level by level in one workgroup,
// in VectorOps' order, into out[v]. The first level's chunks go to the workgroup's waves
// (red_threads: one wave per chunk, at most kRedWaves; their totals in LDS); wave 0 sums those
// (one chunk: fewer than 2^31 entries have at most kRedTot first-level chunks). The same bits as
// one wave walking the levels in turn.
constexpr int kRedWaves = 8, kRedThreads = kRedWaves * kLanes, kRedTot = 512;
static_assert(static_cast<int64_t>(kRedTot) * kChunk * kChunk >= (int64_t(1) << 31), "first-level totals of 2^31 entries");
// the reduction's workgroup for n entries: a wave per first-level chunk of the n / 2048 partials
inline dim3 red_threads(int64_t n) {
  const int64_t c = chunks(chunks(n));
  return dim3(static_cast<unsigned>(kLanes * (c < 1 ? 1 : c > kRedWaves ? kRedWaves : c)));
}
__global__ __launch_bounds__(kRedThreads) void reduce_kernel(int64_t npart, int nv, const double* __restrict__ partial,
                                                             const int32_t* done, double* out) {
  if (done && *done) return;
  __shared__ double tot[2][kRedTot];
  __shared__ double row[kRedWaves][kLanes];
  const int l = threadIdx.x % kLanes, w = threadIdx.x / kLanes;
  const int64_t nch = chunks(npart);
  double total[2] = {0.0, 0.0};
  if (npart > 1) {
    for (int v = 0; v < nv; ++v)
      for (int64_t c = w; c < nch; c += static_cast<int64_t>(blockDim.x / kLanes)) {
        const int64_t begin = c * kChunk;
        const double t =
            wave_chunk_sum(partial + v, nv, begin, npart - begin < kChunk ? npart - begin : kChunk, l, row[w]);
        if (l == 0) tot[v][c] = t;
      }
    __syncthreads();
    if (w == 0)
      for (int v = 0; v < nv; ++v) total[v] = nch > 1 ? wave_chunk_sum(tot[v], 1, 0, nch, l, row[0]) : tot[v][0];
  } else {
    for (int v = 0; v < nv; ++v) total[v] = partial[v];
  }
  if (threadIdx.x != 0) return;
  for (int v = 0; v < nv; ++v) out[v] = total[v];
}

// r = b - A x (ap holds A x); START: also z = inv r, p = z, and the chunk partials of r.r and r.z
// (interleaved); else of r.r alone.
template <typename T, bool START>
__global__ __launch_bounds__(kVecThreads) void residual_kernel(int64_t n, const T* __restrict__ b,
                                                               const T* __restrict__ ap, const T* __restrict__ inv,
                                                               T* __restrict__ r, T* __restrict__ z, T* __restrict__ p,
                                                               double* __restrict__ partial) {
  __shared__ T rs[kChunk], zs[START ? kChunk : 1];
  __shared__ double row[2][kLanes];
  const int64_t begin = static_cast<int64_t>(blockIdx.x) * kChunk;
  const int len = static_cast<int>(n - begin < kChunk ? n - begin : kChunk);
  const int t = threadIdx.x;
  T bv[kPerThread], av[kPerThread], iv[kPerThread];
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    const int k = t + j * kVecThreads;
    const int64_t i = begin + (k < len ? k : 0);
    bv[j] = b[i];
    av[j] = ap[i];
    if constexpr (START) iv[j] = inv[i];
  }
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    const int k = t + j * kVecThreads;
    const T rj = bv[j] + T(-1) * av[j];
    rs[k] = rj;
    if (k < len) r[begin + k] = rj;
    if constexpr (START) {
      const T zj = iv[j] * rj;
      zs[k] = zj;
      if (k < len) {
        z[begin + k] = zj;
        p[begin + k] = zj;
      }
    }
  }
  __syncthreads();
  const int w = t / kLanes, l = t % kLanes;
  if (w >= (START ? 2 : 1)) return;
  double s;
  if constexpr (START) s = wave_staged_dot(rs, w == 0 ? rs : zs, len, l, row[w]);
  else s = wave_staged_dot(rs, rs, len, l, row[w]);
  if (l == 0) partial[(START ? 2 : 1) * static_cast<int64_t>(blockIdx.x) + w] = s;
}

// The solve's state from ||b||, the first residual and r.z (cg.cpp:30-43): one workgroup.
__global__ __launch_bounds__(kVecThreads) void cg_start_kernel(int64_t nb, const double* __restrict__ bpart, int64_t nr,
                                                               const double* __restrict__ rpart, double rtol, double atol,
                                                               int32_t max_it, const int32_t* zeros, CgState* st,
                                                               CgMirror* mirror) {
  __shared__ double row[3][kLanes];
  __shared__ double tot[3];
  const int w = threadIdx.x / kLanes, l = threadIdx.x % kLanes;
  if (w < 3) {
    const double s = w == 0 ? wave_total(bpart, 1, 0, nb, l, row[w]) : wave_total(rpart, 2, w - 1, nr, l, row[w]);
    if (l == 0) tot[w] = s;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  st->rhs_norm = sqrt(tot[0]);
  st->tol = fmax(rtol * st->rhs_norm, atol);
  st->init_res = st->final_res = sqrt(tot[1]);
  st->rz = st->rz_next = tot[2];
  st->beta = 0.0;
  st->it = 0;
  st->max_it = max_it;
  st->indefinite = 0;
  st->zeros = zeros ? *zeros : 0;
  st->converged = st->init_res <= st->tol;
  st->done = st->converged || max_it <= 0 || st->zeros > 0;
  if (st->done) mirror_stop(mirror, st, st->final_res, 0, st->converged);
}

// alpha = r.z / p.Ap from the chunk partials of p.Ap; x += alpha p, r -= alpha Ap, z = inv r
// (cg.cpp:48-64), and the chunk partials of r.r and r.z from the updated values. One workgroup
// per chunk, its loads issued before the total of p.Ap is needed. 27,744 entries: 8.2 -> 4 us and
// one launch less; HBM-bound from about a million entries.
template <typename T>
__global__ __launch_bounds__(kVecThreads) void update_dot_kernel(int64_t n, CgState* st, int64_t npap,
                                                                 const double* __restrict__ pap, T* __restrict__ x,
                                                                 T* __restrict__ r, T* __restrict__ z,
                                                                 const T* __restrict__ p, const T* __restrict__ ap,
                                                                 const T* __restrict__ inv, double* __restrict__ partial,
                                                                 CgMirror* mirror) {
  __shared__ T rs[kChunk], zs[kChunk];
  __shared__ double row[2][kLanes];
  __shared__ double total;
  const int stopped = st->done;
  const double rz = st->rz_next;
  const int64_t begin = static_cast<int64_t>(blockIdx.x) * kChunk;
  const int len = static_cast<int>(n - begin < kChunk ? n - begin : kChunk);
  const int t = threadIdx.x, w = t / kLanes, l = t % kLanes;
  T xv[kPerThread], rv[kPerThread], pv[kPerThread], av[kPerThread], iv[kPerThread];
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    const int k = t + j * kVecThreads;
    const int64_t i = begin + (k < len ? k : 0);
    xv[j] = x[i];
    rv[j] = r[i];
    pv[j] = p[i];
    av[j] = ap[i];
    iv[j] = inv[i];
  }
  if (w == 0) {
    const double s = wave_total(pap, 1, 0, npap, l, row[0]);
    if (l == 0) total = s;
  }
  if (stopped) return;
  __syncthreads();
  if (!(total > 0.0)) {  // p.Ap <= 0: the operator is not positive definite (cg.cpp:49-53)
    if (blockIdx.x == 0 && t == 0) {
      st->indefinite = 1;
      st->done = 1;
      mirror_stop(mirror, st, st->final_res, st->it, 0);
    }
    return;
  }
  const T alpha = static_cast<T>(rz / total);
  if (blockIdx.x == 0 && t == 0) {
    st->rz = rz;
    st->it += 1;
  }
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    const int k = t + j * kVecThreads;
    const T xj = xv[j] + alpha * pv[j];
    const T rj = rv[j] + (-alpha) * av[j];
    const T zj = iv[j] * rj;
    rs[k] = rj;
    zs[k] = zj;
    if (k < len) {
      x[begin + k] = xj;
      r[begin + k] = rj;
      z[begin + k] = zj;
    }
  }
  __syncthreads();
  if (w >= 2) return;
  const double s = wave_staged_dot(rs, w == 0 ? rs : zs, len, l, row[w]);
  if (l == 0) partial[2 * static_cast<int64_t>(blockIdx.x) + w] = s;
}

// The stop test on ||r|| (cg.cpp:60) and p = z + beta p (cg.cpp:68) from the chunk partials of r.r
// and r.z, for products that take p as it is (launch_box_cg's form it themselves). The loads are
// issued before the stop flag is read: one round of memory latency, not two.
template <typename T>
__global__ __launch_bounds__(kVecThreads) void direction_kernel(int64_t n, CgDirection<T> d) {
  __shared__ double row[2][kLanes];
  __shared__ double tot[2];
  __shared__ int32_t stopped;  // one thread reads the flag: another workgroup may be setting it (cg_decide)
  const int64_t begin = static_cast<int64_t>(blockIdx.x) * kChunk;
  const int len = static_cast<int>(n - begin < kChunk ? n - begin : kChunk);
  const int t = threadIdx.x, w = t / kLanes, l = t % kLanes;
  const int it = d.st->it, max_it = d.st->max_it;
  const int done = t == 0 ? d.st->done : 0;
  const double rz = d.st->rz, tol = d.st->tol;
  T zv[kPerThread], pv[kPerThread];
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    const int k = t + j * kVecThreads;
    const int64_t i = begin + (k < len ? k : 0);
    zv[j] = d.z[i];
    pv[j] = d.p_old[i];
  }
  if (w < 2) {
    const double s = wave_total(d.part, 2, w, d.npart, l, row[w]);
    if (l == 0) tot[w] = s;
    if (t == 0) stopped = done;
  }
  __syncthreads();
  if (stopped) return;
  double beta;
  if (!cg_decide(d.st, d.mirror, it, max_it, tol, rz, tot[0], tot[1], blockIdx.x == 0 && t == 0, beta)) return;
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    const int k = t + j * kVecThreads;
    if (k < len) d.p[begin + k] = zv[j] + static_cast<T>(beta) * pv[j];
  }
}

template <typename T>
__global__ void reciprocal_kernel(int64_t n, const double* __restrict__ d, T* __restrict__ inv, int32_t* zeros) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) {
    if (d[i] == 0.0) atomicAdd(zeros, 1);
    inv[i] = static_cast<T>(1.0 / d[i]);
  }
}

// x64 += scale * d32; r32 = scale_in * r64 (conversions of the refinement)
__global__ void refine_update_kernel(int64_t n, double* __restrict__ x, const float* __restrict__ d, double s) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) x[i] += s * static_cast<double>(d[i]);
}
__global__ void to_f32_kernel(int64_t n, const double* __restrict__ a, float* __restrict__ b, double s) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) b[i] = static_cast<float>(a[i] * s);
}
template <typename T>
__global__ void zero_kernel(int64_t n, T* __restrict__ a) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) a[i] = T(0);
}

// Plain vector copy (also the calibration kernel of the HBM traffic counters: it moves exactly
// n * 16 bytes).
__global__ void copy_kernel(int64_t n, const double* __restrict__ a, double* __restrict__ b) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

int copy64(fx_ctx* ctx, int64_t n, const double* a, double* b) {
  if (n <= 0) return FX_OK;
  hipLaunchKernelGGL(copy_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, ctx->stream, n, a, b);
  FX_HIP(ctx, hipGetLastError());
  FX_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return FX_OK;
}

namespace {

inline dim3 grid_of(int64_t n, int bs = 256) { return dim3(static_cast<unsigned>((n + bs - 1) / bs)); }
inline dim3 chunk_grid(int64_t n) { return dim3(static_cast<unsigned>(chunks(n))); }

// Reduction scratch: the chunk partials of one dot, then of two, then their totals.
int ensure_red(fx_ctx* ctx, int64_t n) {
  const size_t need = cg_red_doubles(n);
  if (ctx->red_cap >= need) return FX_OK;
  release_cg_graphs(ctx, nullptr);  // captured graphs read the old buffer
  if (ctx->red) (void)hipFree(ctx->red);
  ctx->red = nullptr;
  FX_HIP(ctx, hipMalloc(&ctx->red, need * sizeof(double)));
  ctx->red_cap = need;
  return FX_OK;
}

}  // namespace

int dot64(fx_ctx* ctx, int64_t n, const double* x, const double* y, double* out) {
  if (n <= 0) {
    *out = 0.0;
    return FX_OK;
  }
  if (int rc = ensure_red(ctx, n)) return rc;
  double* dres = static_cast<double*>(ctx->host_pinned);  // the device writes the total to host memory
  hipLaunchKernelGGL(chunk_dot_kernel<double>, chunk_grid(n), dim3(kVecThreads), 0, ctx->stream, n, x, y, ctx->red,
                     static_cast<const int32_t*>(nullptr));
  hipLaunchKernelGGL(reduce_kernel, dim3(1), red_threads(n), 0, ctx->stream, chunks(n), 1, ctx->red,
                     static_cast<const int32_t*>(nullptr), dres);
  FX_HIP(ctx, hipGetLastError());
  FX_HIP(ctx, hipStreamSynchronize(ctx->stream));
  *out = *dres;
  return FX_OK;
}

void release_cg_graphs(fx_ctx* ctx, const void* owner) {
  auto& g = ctx->cg_graphs;
  for (auto it = g.begin(); it != g.end();) {
    if (owner && it->owner != owner) {
      ++it;
      continue;
    }
    if (it->exec) (void)hipGraphExecDestroy(it->exec);
    if (it->graph) (void)hipGraphDestroy(it->graph);
    it = g.erase(it);
  }
}

namespace {

constexpr int kGraphIters = 8;     // CG iterations per captured graph
constexpr size_t kMaxGraphs = 64;  // per context (a serving worker keeps a few dozen block sizes)

struct CgGraphKey {
  const void* owner;
  int64_t n;
  int32_t tsize, initial;
  double ks, kd, km, rtol, atol;
  const void* ptr[11];
  // the batch arrays the operator kernels read whose pointers change between calls: the
  // committed and trial histories swap on every commit (the committed tangent is formed from
  // the committed history), so each parity of the swap has its own graph
  const void* state[2];
};

// The captured graph of kGraphIters iterations for this key, capturing it on first use.
template <typename Body>
hipGraphExec_t cg_graph(fx_ctx* ctx, const CgGraphKey& key, Body body) {
  std::vector<unsigned char> k(sizeof key);
  std::memcpy(k.data(), &key, sizeof key);
  for (auto& g : ctx->cg_graphs)
    if (g.key == k) return g.exec;
  if (ctx->cg_graphs.size() >= kMaxGraphs) {  // drop the oldest
    fx_cg_graph& old = ctx->cg_graphs.front();
    if (old.exec) (void)hipGraphExecDestroy(old.exec);
    if (old.graph) (void)hipGraphDestroy(old.graph);
    ctx->cg_graphs.erase(ctx->cg_graphs.begin());
  }
  hipStream_t s = ctx->stream;
  if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess) return nullptr;
  int rc = FX_OK;
  for (int i = 0; i < kGraphIters && rc == FX_OK; ++i) rc = body(i);
  hipGraph_t graph = nullptr;
  const hipError_t ec = hipStreamEndCapture(s, &graph);
  hipGraphExec_t exec = nullptr;
  if (rc != FX_OK || ec != hipSuccess || !graph || hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess) {
    if (graph) (void)hipGraphDestroy(graph);
    (void)hipGetLastError();
    return nullptr;  // the caller launches the iterations itself
  }
  ctx->cg_graphs.push_back(fx_cg_graph{std::move(k), key.owner, graph, exec});
  return exec;
}

// A dot's chunk partials as the kernels that need their total take them: the partials themselves,
// or past kInlineParts the total(s), reduced by a launch of their own (into tot).
struct Parts {
  int64_t n;
  const double* p;
};
Parts total_of(fx_ctx* ctx, int64_t n, int nv, const double* part, double* tot, const int32_t* done) {
  if (chunks(n) <= kInlineParts) return Parts{chunks(n), part};
  hipLaunchKernelGGL(reduce_kernel, dim3(1), red_threads(n), 0, ctx->stream, chunks(n), nv, part, done, tot);
  return Parts{1, tot};
}

// A CG solve's device arrays (solver numbering) and the operator they belong to.
template <typename T>
struct CgVectors {
  const T *inv, *b;
  T *x, *r, *z, *p, *p2, *ap;  // p2: the direction's second buffer (products that form it)
  CgState* st;
  double* red;       // cg_red_doubles(n)
  CgMirror* mirror;  // or null
};

// The CG setup on the device: ||b||, r = b - A x, z = inv r, p = z, r.z. zeros: the count of zero
// diagonal entries (a solve that has any stops before its first iteration), or null.
template <typename T, typename Op>
int cg_setup(fx_ctx* ctx, int64_t n, const Op& op, const CgVectors<T>& v, double rtol, double atol, int max_it,
             const int32_t* zeros) {
  hipStream_t s = ctx->stream;
  double *p1 = v.red, *p2 = v.red + chunks(n), *tot = v.red + 3 * chunks(n);
  const int32_t* always = nullptr;
  hipLaunchKernelGGL(chunk_dot_kernel<T>, chunk_grid(n), dim3(kVecThreads), 0, s, n, v.b, v.b, p1, always);
  const Parts bb = total_of(ctx, n, 1, p1, tot, always);
  if (int rc = op.apply(v.x, v.ap)) return rc;
  hipLaunchKernelGGL((residual_kernel<T, true>), chunk_grid(n), dim3(kVecThreads), 0, s, n, v.b, v.ap, v.inv, v.r, v.z,
                     v.p, p2);
  const Parts rr = total_of(ctx, n, 2, p2, tot + 1, always);
  hipLaunchKernelGGL(cg_start_kernel, dim3(1), dim3(kVecThreads), 0, s, bb.n, bb.p, rr.n, rr.p, rtol, atol, max_it,
                     zeros, v.st, v.mirror);
  FX_HIP(ctx, hipGetLastError());
  return FX_OK;
}

// One CG iteration (cg.cpp:44-69): A p with p.Ap, then the x, r, z update with r.r and r.z; a no-op
// once the state's stop flag is set. The stop test and the next direction follow the update
// (direction_kernel), or lead the next iteration's product where the operator forms its direction
// itself: iteration i then writes p into buffer i mod 2. last: the stop test also runs by itself
// (no iteration follows, or not before the host has looked).
template <typename T, typename Op>
int cg_iteration(fx_ctx* ctx, int64_t n, const Op& op, const CgVectors<T>& v, int i, bool last) {
  hipStream_t s = ctx->stream;
  double *p1 = v.red, *p2 = v.red + chunks(n), *tot = v.red + 3 * chunks(n);
  const int32_t* done = &v.st->done;
  const bool own = op.own_direction();
  T* p = own && (i & 1) ? v.p2 : v.p;
  if (own) {
    const CgDirection<T> d{v.st, v.mirror, chunks(n), p2, v.z, (i & 1) ? v.p : v.p2, p};
    if (int rc = op.apply_dot(d, v.ap, p1)) return rc;
  } else if (int rc = op.apply_dot(p, v.ap, p1, v.st)) {
    return rc;
  }
  const Parts pap = total_of(ctx, n, 1, p1, tot, done);
  hipLaunchKernelGGL(update_dot_kernel<T>, chunk_grid(n), dim3(kVecThreads), 0, s, n, v.st, pap.n, pap.p, v.x, v.r, v.z,
                     p, v.ap, v.inv, p2, v.mirror);
  const Parts rr = total_of(ctx, n, 2, p2, tot + 1, done);
  if (!own)
    hipLaunchKernelGGL(direction_kernel<T>, chunk_grid(n), dim3(kVecThreads), 0, s, n,
                       CgDirection<T>{v.st, v.mirror, rr.n, rr.p, v.z, p, p});
  else if (last)  // the decision alone: no entry of p
    hipLaunchKernelGGL(direction_kernel<T>, dim3(1), dim3(kVecThreads), 0, s, static_cast<int64_t>(0),
                       CgDirection<T>{v.st, v.mirror, rr.n, rr.p, v.z, p, p});
  return FX_OK;
}

// K_eff of a batch for vector type T: y = A x, and A p with the chunk partials of p.Ap.
template <typename T>
struct BatchOp {
  fx_batch* b;
  fx_coeffs k;
  int apply(const T* x, T* y) const {
    if constexpr (sizeof(T) == 8) return operator_apply64(b, k, x, y, nullptr);
    else return operator_apply32(b, k, x, y, nullptr);
  }
  bool own_direction() const { return box_forms_direction(b); }
  int apply_dot(const CgDirection<T>& d, T* ap, double* part) const { return launch_box_cg<T>(b, k, d, ap, part); }
  int apply_dot(T* p, T* ap, double* part, CgState* st) const {
    if (box_sums_with_dot(b)) return apply_dot(CgDirection<T>{st, nullptr, 0, nullptr, nullptr, nullptr, p}, ap, part);
    const int32_t* done = &st->done;
    int rc;
    if constexpr (sizeof(T) == 8) rc = operator_apply64(b, k, p, ap, done);
    else rc = operator_apply32(b, k, p, ap, done);
    if (rc) return rc;
    hipLaunchKernelGGL(chunk_dot_kernel<T>, chunk_grid(b->neq), dim3(kVecThreads), 0, b->ctx->stream, b->neq, p, ap, part,
                       done);
    return FX_OK;
  }
};

// The captured graph of a solve's iterations (null: graphs off, or the capture failed).
template <typename T>
hipGraphExec_t cg_solve_graph(fx_ctx* ctx, int64_t n, const CgVectors<T>& v, double rtol, double atol, int max_it,
                              const BatchOp<T>& op) {
  if (!ctx->use_graphs || max_it <= 0) return nullptr;
  const fx_batch* owner = op.b;
  CgGraphKey key{};
  key.owner = owner;
  key.n = n;
  key.tsize = static_cast<int32_t>(sizeof(T));
  key.initial = op.k.initial;
  key.ks = op.k.stiffness;
  key.kd = op.k.damping;
  key.km = op.k.mass;
  key.rtol = rtol;
  key.atol = atol;
  const void* ptrs[11] = {v.inv, v.b, v.x, v.r, v.z, v.p, v.p2, v.ap, v.st, v.red, v.mirror};
  for (int i = 0; i < 11; ++i) key.ptr[i] = ptrs[i];
  key.state[0] = owner->state_c;
  key.state[1] = owner->state_t;
  return cg_graph(ctx, key, [&](int i) -> int { return cg_iteration<T>(ctx, n, op, v, i, i + 1 == kGraphIters); });
}

// The CG iterations on the device after cg_setup: the host launches them while it watches the
// solve's mirror. With graphs on, each group replays a captured graph of kGraphIters iterations
// (the same kernels and arguments, so the same bits as launching them).
template <typename T>
int cg_device(fx_ctx* ctx, int64_t n, const BatchOp<T>& op, const T* inv, const T* b, T* x, T* r, T* z, T* p, T* p2,
              T* ap, CgState* st, double rtol, double atol, int max_it, const int32_t* zeros, CgMirror& host) {
  if (int rc = ensure_red(ctx, n)) return rc;
  // the mirror sits behind the dots' result in the context's pinned block
  CgMirror* mirror = reinterpret_cast<CgMirror*>(static_cast<char*>(ctx->host_pinned) + 256);
  __atomic_store_n(&mirror->it, 0, __ATOMIC_RELAXED);
  __atomic_store_n(&mirror->done, 0, __ATOMIC_RELEASE);
  const CgVectors<T> v{inv, b, x, r, z, p, p2, ap, st, ctx->red, mirror};
  if (int rc = cg_setup<T>(ctx, n, op, v, rtol, atol, max_it, zeros)) return rc;
  hipGraphExec_t exec = cg_solve_graph<T>(ctx, n, v, rtol, atol, max_it, op);
  struct Device {  // cg_watch's device: this solve
    fx_ctx* ctx;
    CgMirror* mirror;
    hipGraphExec_t exec;
    const CgVectors<T>& v;
    const BatchOp<T>& op;
    int64_t n;
    int max_it;
    int it() const { return __atomic_load_n(&mirror->it, __ATOMIC_RELAXED); }
    bool done() const { return __atomic_load_n(&mirror->done, __ATOMIC_ACQUIRE) != 0; }
    int launch(int i) {
      if (exec) {
        FX_HIP(ctx, hipGraphLaunch(exec, ctx->stream));
        return FX_OK;
      }
      if (int rc = cg_iteration<T>(ctx, n, op, v, i, i + 1 == max_it)) return rc;
      FX_HIP(ctx, hipGetLastError());
      return FX_OK;
    }
    int idle(bool& is) {
      const hipError_t q = hipStreamQuery(ctx->stream);
      is = q == hipSuccess;
      if (q != hipErrorNotReady) FX_HIP(ctx, q);
      return FX_OK;
    }
    int stalled() {
      ctx->error = "CG: the device did not report the queued iterations";
      return FX_EDEVICE;
    }
  } dev{ctx, mirror, exec, v, op, n, max_it};
  if (int rc = cg_watch(dev, max_it, exec ? kGraphIters : 1)) return rc;
  host = *mirror;
  return FX_OK;
}

// The Jacobi preconditioner 1 / diag(K_eff), queued; the count of zero entries in *zeros (device).
int jacobi_queue(fx_batch* b, const fx_coeffs& k, double* d, void* inv, bool f32, int32_t** zeros) {
  fx_ctx* ctx = b->ctx;
  if (int rc = operator_diagonal64(b, k, d)) return rc;
  int32_t* z = reinterpret_cast<int32_t*>(ctx->scalars) + 64;
  FX_HIP(ctx, hipMemsetAsync(z, 0, sizeof(int32_t), ctx->stream));
  if (f32)
    hipLaunchKernelGGL(reciprocal_kernel<float>, grid_of(b->neq), dim3(256), 0, ctx->stream, b->neq, d,
                       static_cast<float*>(inv), z);
  else
    hipLaunchKernelGGL(reciprocal_kernel<double>, grid_of(b->neq), dim3(256), 0, ctx->stream, b->neq, d,
                       static_cast<double*>(inv), z);
  FX_HIP(ctx, hipGetLastError());
  *zeros = z;
  return FX_OK;
}

int zero_diagonal(fx_ctx* ctx, int32_t zeros) {
  ctx->error = "Jacobi: " + std::to_string(zeros) + " zero diagonal entries";
  return FX_EZERO;
}

int jacobi_inverse(fx_batch* b, const fx_coeffs& k, double* d, void* inv, bool f32) {
  fx_ctx* ctx = b->ctx;
  int32_t *zeros = nullptr, hz = 0;
  if (int rc = jacobi_queue(b, k, d, inv, f32, &zeros)) return rc;
  FX_HIP(ctx, hipMemcpyAsync(&hz, zeros, sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
  FX_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return hz > 0 ? zero_diagonal(ctx, hz) : FX_OK;
}

// ||b - A x|| in FP64, queued; its chunk partials reduced into the context's pinned block, which
// holds the square once the stream is idle.
int queue_residual_norm(fx_batch* b, const fx_coeffs& k, const double* bi, const double* xi, double* ap, double* r) {
  fx_ctx* ctx = b->ctx;
  const int64_t n = b->neq;
  if (int rc = ensure_red(ctx, n)) return rc;
  if (int rc = operator_apply64(b, k, xi, ap)) return rc;
  double* nul = nullptr;
  hipLaunchKernelGGL((residual_kernel<double, false>), chunk_grid(n), dim3(kVecThreads), 0, ctx->stream, n, bi, ap,
                     static_cast<const double*>(nullptr), r, nul, nul, ctx->red);
  hipLaunchKernelGGL(reduce_kernel, dim3(1), red_threads(n), 0, ctx->stream, chunks(n), 1, ctx->red,
                     static_cast<const int32_t*>(nullptr), static_cast<double*>(ctx->host_pinned));
  FX_HIP(ctx, hipGetLastError());
  return FX_OK;
}
// A solve's end: the true residual, x back to the caller's numbering, both in place on return.
int finish_solve(fx_batch* b, const fx_coeffs& k, const double* bi, const double* xi, double* ap, double* r, double* x,
                 fx_solve_result& res) {
  if (int rc = queue_residual_norm(b, k, bi, xi, ap, r)) return rc;
  if (int rc = to_external<double>(b, xi, x)) return rc;
  FX_HIP(b->ctx, hipStreamSynchronize(b->ctx->stream));
  res.true_residual = std::sqrt(*static_cast<const double*>(b->ctx->host_pinned));
  return FX_OK;
}

void cg_result(const CgMirror& h, fx_solve_result& res) {
  res = fx_solve_result{};
  res.converged = h.converged;
  res.iterations = h.it;
  res.indefinite = h.indefinite;
  res.rhs_norm = h.rhs_norm;
  res.initial_residual = h.init_res;
  res.final_residual = h.final_res;
}

}  // namespace

int jacobi_inverse_public(fx_batch* b, const fx_coeffs& k, double* d, double* inv) {
  return jacobi_inverse(b, k, d, inv, false);
}

// CG + Jacobi on vectors already in the solver numbering (no permutation, no true residual).
int cg64_solver(fx_batch* b, const fx_coeffs& k, const fx_solve_options& o, const double* bi, double* xi,
                fx_solve_result& res) {
  fx_ctx* ctx = b->ctx;
  const int64_t n = b->neq;
  double *r = b->work, *z = r + n, *p = z + n, *ap = p + n, *inv = ap + n, *d = inv + n;
  int32_t* zeros = nullptr;
  if (int rc = jacobi_queue(b, k, d, inv, false, &zeros)) return rc;
  CgMirror h{};
  if (int rc = cg_device<double>(ctx, n, BatchOp<double>{b, k}, inv, bi, xi, r, z, p, d, ap,
                                 static_cast<CgState*>(ctx->scalars), o.relative_tolerance, o.absolute_tolerance,
                                 o.max_iterations, zeros, h))
    return rc;
  if (h.zeros > 0) return zero_diagonal(ctx, h.zeros);
  cg_result(h, res);
  return FX_OK;
}

int cg64(fx_batch* b, const fx_coeffs& k, const fx_solve_options& o, const double* rhs, double* x,
         fx_solve_result& res) {
  const int64_t n = b->neq;
  double *r = b->work, *ap = r + 3 * n, *bi = r + 6 * n, *xi = r + 7 * n;
  if (int rc = to_internal<double>(b, rhs, bi)) return rc;
  if (int rc = to_internal<double>(b, x, xi)) return rc;
  if (int rc = cg64_solver(b, k, o, bi, xi, res)) return rc;
  return finish_solve(b, k, bi, xi, ap, r, x, res);
}

size_t cg_red_doubles(int64_t n) { return static_cast<size_t>(3 * chunks(n) + 16); }

// Several FP64 CG solves advanced together on one stream (the serving loop's admission round): each
// poll round launches every unfinished solve's next group of iterations (a captured graph per
// solve with graphs on) and then reads every solve's state with one synchronisation. A solve
// keeps its own state block and reduction scratch (the batch's), and its kernels, arguments and
// order are those of cg64 on its own batch, so its iterates, result and x are the same bits.
int cg64_many(int32_t nb, fx_batch* const* bs, const fx_coeffs& k, const fx_solve_options& o,
              const double* const* rhs, double* const* x, fx_solve_result* res) {
  if (nb <= 0) return FX_OK;
  fx_ctx* ctx = bs[0]->ctx;
  hipStream_t s = ctx->stream;
  struct Solve {
    CgVectors<double> v;
    double *bi, *xi;
    hipGraphExec_t exec;
    int launched;
    bool active;
  };
  std::vector<Solve> sv(static_cast<size_t>(nb));
  std::vector<CgState> host(static_cast<size_t>(nb));
  for (int32_t i = 0; i < nb; ++i) {
    fx_batch* b = bs[i];
    const int64_t n = b->neq;
    double *r = b->work, *inv = r + 4 * n, *bi = r + 6 * n, *xi = r + 7 * n;
    sv[i] = Solve{CgVectors<double>{inv, bi, xi, r, r + n, r + 2 * n, r + 5 * n, r + 3 * n, reinterpret_cast<CgState*>(b->cg_state),
                                    b->cg_red, nullptr},
                  bi, xi, nullptr, 0, true};
    if (int rc = to_internal<double>(b, rhs[i], bi)) return rc;
    if (int rc = to_internal<double>(b, x[i], xi)) return rc;
    if (int rc = jacobi_inverse(b, k, r + 5 * n, inv, false)) return rc;
    const BatchOp<double> op{b, k};
    if (int rc = cg_setup<double>(ctx, n, op, sv[i].v, o.relative_tolerance, o.absolute_tolerance, o.max_iterations,
                                  nullptr))
      return rc;
    sv[i].exec = cg_solve_graph<double>(ctx, n, sv[i].v, o.relative_tolerance, o.absolute_tolerance, o.max_iterations,
                                        op);
  }
  const int max_it = o.max_iterations;
  for (int poll = 4, left = nb; left > 0; poll = std::min(poll * 2, 64)) {
    for (int32_t i = 0; i < nb; ++i)
      if (sv[i].active)
        FX_HIP(ctx, hipMemcpyAsync(&host[i], sv[i].v.st, sizeof(CgState), hipMemcpyDeviceToHost, s));
    FX_HIP(ctx, hipStreamSynchronize(s));
    for (int32_t i = 0; i < nb; ++i) {
      Solve& v = sv[i];
      if (!v.active) continue;
      fx_batch* b = bs[i];
      const CgState& h = host[i];
      if (h.done || v.launched >= max_it) {
        // finished: cg64_solver's result, then cg64's true residual and permutation
        cg_result(CgMirror{h.rhs_norm, h.init_res, h.final_res, h.it, h.converged, h.indefinite, 0, 1, 0}, res[i]);
        if (int rc = finish_solve(b, k, v.bi, v.xi, v.v.ap, v.v.r, x[i], res[i])) return rc;
        v.active = false;
        --left;
        continue;
      }
      const int batch = std::min(poll, max_it - v.launched);
      if (v.exec) {
        const int graphs = (batch + kGraphIters - 1) / kGraphIters;
        for (int g = 0; g < graphs; ++g) FX_HIP(ctx, hipGraphLaunch(v.exec, s));
        v.launched += graphs * kGraphIters;
      } else {
        for (int it = 0; it < batch; ++it)
          if (int rc = cg_iteration<double>(ctx, b->neq, BatchOp<double>{b, k}, v.v, v.launched + it, it + 1 == batch))
            return rc;
        v.launched += batch;
      }
      FX_HIP(ctx, hipGetLastError());
    }
  }
  return FX_OK;
}

// GMRES (method 1) or CG with the GMRES fallback (method 2) at the C ABI: permutations around
// the solver-numbering solve, the true residual reported.
int krylov64(fx_batch* b, int method, const fx_coeffs& k, const fx_solve_options& o, const double* rhs, double* x,
             fx_solve_result& res) {
  const int64_t n = b->neq;
  double *r = b->work, *ap = r + 3 * n, *bi = r + 6 * n, *xi = r + 7 * n;
  if (int rc = to_internal<double>(b, rhs, bi)) return rc;
  if (int rc = to_internal<double>(b, x, xi)) return rc;
  if (int rc = method == 1 ? gmres64_solver(b, k, o, bi, xi, res) : krylov64_solver(b, k, o, bi, xi, res)) return rc;
  return finish_solve(b, k, bi, xi, ap, r, x, res);
}

int cg_mixed(fx_batch* b, const fx_coeffs& k, const fx_solve_options& o, double inner_rtol, const double* rhs,
             double* x, fx_solve_result& res) {
  const int64_t n = b->neq;
  double *bi = b->work + 6 * n, *xi = b->work + 7 * n;
  if (int rc = to_internal<double>(b, rhs, bi)) return rc;
  if (int rc = to_internal<double>(b, x, xi)) return rc;
  if (int rc = cg_mixed_solver(b, k, o, inner_rtol, bi, xi, res)) return rc;
  if (int rc = to_external<double>(b, xi, x)) return rc;
  FX_HIP(b->ctx, hipStreamSynchronize(b->ctx->stream));
  return FX_OK;
}

int cg_mixed_solver(fx_batch* b, const fx_coeffs& k, const fx_solve_options& o, double inner_rtol, const double* bi,
                    double* xi, fx_solve_result& res) {
  fx_ctx* ctx = b->ctx;
  if (!b->has_f32) {
    ctx->error = "fx_cg_mixed: the batch was created without FX_BATCH_FP32";
    return FX_EUNSUP;
  }
  const int64_t n = b->neq;
  double *r64 = b->work, *ap64 = r64 + 3 * n, *d64 = r64 + 5 * n;
  float *inv = b->work32, *r = inv + n, *z = r + n, *p = z + n, *ap = p + n, *dx = ap + n, *rhs32 = dx + n,
        *p2 = rhs32 + n;
  if (int rc = jacobi_inverse(b, k, d64, inv, true)) return rc;
  CgState* st = static_cast<CgState*>(ctx->scalars);
  hipStream_t s = ctx->stream;
  double bb = 0;
  if (int rc = dot64(ctx, n, bi, bi, &bb)) return rc;
  const double bnorm = std::sqrt(bb);
  const double tol = std::max(o.relative_tolerance * bnorm, o.absolute_tolerance);
  res = fx_solve_result{};
  res.rhs_norm = bnorm;
  int total_inner = 0;
  for (int outer = 0;; ++outer) {
    // r = b - A x in FP64
    if (int rc = queue_residual_norm(b, k, bi, xi, ap64, r64)) return rc;
    FX_HIP(ctx, hipStreamSynchronize(s));
    const double rn = std::sqrt(*static_cast<const double*>(ctx->host_pinned));
    if (outer == 0) res.initial_residual = rn;
    res.final_residual = res.true_residual = rn;
    res.outer_iterations = outer;
    if (rn <= tol) {
      res.converged = 1;
      break;
    }
    if (total_inner >= o.max_iterations || outer >= 100) break;
    // inner FP32 solve of A d = r / ||r||
    hipLaunchKernelGGL(to_f32_kernel, grid_of(n), dim3(256), 0, s, n, r64, rhs32, 1.0 / rn);
    hipLaunchKernelGGL(zero_kernel<float>, grid_of(n), dim3(256), 0, s, n, dx);
    CgMirror h{};
    if (int rc = cg_device<float>(ctx, n, BatchOp<float>{b, k}, inv, rhs32, dx, r, z, p, p2, ap, st, inner_rtol, 0.0,
                                  o.max_iterations - total_inner, nullptr, h))
      return rc;
    total_inner += h.it;
    if (h.indefinite) res.indefinite = 1;
    hipLaunchKernelGGL(refine_update_kernel, grid_of(n), dim3(256), 0, s, n, xi, dx, rn);
    FX_HIP(ctx, hipGetLastError());
    if (h.it == 0) break;  // no progress possible
  }
  res.iterations = total_inner;
  return FX_OK;
}

}  // namespace fx

// ---- VectorOps::dot without allocation (fx_dot_static) ------------------------------------
// The reduction scratch of fx_dot_static: a fixed array of the library on every device it runs
// on, sized for FX_DOT_STATIC_MAX_N entries (one chunk partial per 2048 entries, then the level
// buffers reduce_kernel walks: 131,220 doubles, 1.05 MB). In host code `scratch` names a host
// stand-in, never the device memory: host code uses only the address hipGetSymbolAddress gives
// for the current device, kept per device in scratch_ptr.
namespace fx {
namespace {

constexpr int64_t kStaticDotChunks = FX_DOT_STATIC_MAX_N / kChunk;
constexpr size_t kStaticScratch = kStaticDotChunks + 2 * (kStaticDotChunks / kChunk + 2) + 16;
static_assert(FX_DOT_STATIC_MAX_N % kChunk == 0, "whole chunks");

static __device__ __align__(256) double scratch[kStaticScratch];

constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
double* scratch_ptr[kMaxDevices] = {};

__global__ void store_zero_kernel(double* out) {
  if (threadIdx.x == 0 && blockIdx.x == 0) out[0] = 0.0;
}

}  // namespace

// Once per device, with that device current (fx_ctx_create): the device address of the array.
int static_scratch_init(fx_ctx* ctx) {
  if (ctx->device < 0 || ctx->device >= kMaxDevices) {
    ctx->error = "fx_ctx_create: device index beyond the static scratch table";
    return FX_EINVAL;
  }
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (scratch_ptr[ctx->device]) return FX_OK;
  void* p = nullptr;
  FX_HIP(ctx, hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  if (!p) {
    ctx->error = "hipGetSymbolAddress(scratch): null address";
    return FX_EDEVICE;
  }
  scratch_ptr[ctx->device] = static_cast<double*>(p);
  return FX_OK;
}

// The kernels and arguments of dot64 on the device's fixed scratch, the result left in device
// memory: no allocation, no host synchronisation.
int dot64_static(fx_ctx* ctx, int64_t n, const double* x, const double* y, double* out_dev) {
  double* base = nullptr;
  {
    std::lock_guard<std::mutex> lock(scratch_mutex);
    base = scratch_ptr[ctx->device];
  }
  if (!base) {
    ctx->error = "fx_dot_static: no static scratch on this device (context set-up failed)";
    return FX_EDEVICE;
  }
  hipStream_t s = ctx->stream;
  if (n == 0) {
    hipLaunchKernelGGL(store_zero_kernel, dim3(1), dim3(64), 0, s, out_dev);
    FX_HIP(ctx, hipGetLastError());
    return FX_OK;
  }
  hipLaunchKernelGGL(chunk_dot_kernel<double>, dim3(static_cast<unsigned>(chunks(n))), dim3(kVecThreads), 0, s, n, x, y,
                     base, static_cast<const int32_t*>(nullptr));
  hipLaunchKernelGGL(reduce_kernel, dim3(1), red_threads(n), 0, s, chunks(n), 1, base,
                     static_cast<const int32_t*>(nullptr), out_dev);
  FX_HIP(ctx, hipGetLastError());
  return FX_OK;
}

}  // namespace fx

extern "C" int fx_dot_static(fx_ctx* ctx, int64_t n, const double* x, const double* y, double* out_dev) {
  if (!ctx || !out_dev || (n > 0 && (!x || !y))) {
    if (ctx) ctx->error = "fx_dot_static: null argument";
    else fx::set_thread_error("fx_dot_static: null argument");
    return FX_EINVAL;
  }
  if (n < 0 || n > FX_DOT_STATIC_MAX_N) {
    ctx->error = "fx_dot_static: n = " + std::to_string(n) + " outside [0, FX_DOT_STATIC_MAX_N = " +
                 std::to_string(static_cast<int64_t>(FX_DOT_STATIC_MAX_N)) + "]";
    return FX_EINVAL;
  }
  return fx::dot64_static(ctx, n, x, y, out_dev);
}
