// Flexible GMRES(m) with classical Gram-Schmidt run twice (CGS2) and the Jacobi
// preconditioner on the right (src/solvers/gmres.cpp:32-123), and the Krylov driver that runs
// CG and falls back to GMRES from the same initial guess when CG meets p^T A p <= 0
// (src/solvers/krylov.cpp:25-42).
//
// The basis V (m + 1 vectors) and the preconditioned directions Z (m vectors) live in the
// batch's GMRES workspace (FX_BATCH_GMRES). An Arnoldi step stays on the device: its projection
// coefficients are dots in the VectorOps order (BlockOps::dots, block_ops.cpp:59-78) whose totals
// the kernel that subtracts sum_c coef_c V(:, c) (BlockOps::combine :80-92) forms itself, and the
// device writes each Hessenberg column to pinned host memory. The rotations, the stop test and
// the small triangular solve run on the host, which keeps a few steps queued ahead: a step past
// the stop only writes columns that are not used.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "fx_cg_watch.hpp"
#include "fx_internal.hpp"
#include "fx_kernels.hpp"
#include "fx_vecops.hpp"

namespace fx {

namespace {

constexpr int kThreads = 256;
inline dim3 grid(int64_t n) { return dim3(static_cast<unsigned>((n + kThreads - 1) / kThreads)); }

__global__ void gm_residual_kernel(int64_t n, const double* __restrict__ b, const double* __restrict__ w,
                                   double* __restrict__ r) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) r[i] = b[i] + -1.0 * w[i];
}
// The dots of one Gram-Schmidt pass: column c's chunk partials at part + c * stride (npart of them),
// or past kInlineParts their totals (npart = 1, stride = 1).
struct Dots {
  const double* part;
  int64_t npart, stride;
};

// The chunk partial of V(:, col) . w by one wave, in VectorOps' order (w: global or LDS).
__device__ __forceinline__ double wave_chunk_dot(const double* __restrict__ v, const double* w, int len, int l,
                                                 double* row) {
  double s = 0.0;
  for (int k0 = 0; k0 < len; k0 += 16 * kLanes) {
    double a[16], b[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int k = k0 + l + j * kLanes, i = k < len ? k : 0;
      a[j] = v[i];
      b[j] = w[i];
    }
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (k0 + l + j * kLanes < len) s += a[j] * b[j];
  }
  return lane_order_sum(s, l, len < kLanes ? len : kLanes, row);
}

constexpr int kDotWaves = 4;

// The chunk partials of ncol columns' dots with w: a wave per (chunk, column), 32 entries a lane in
// two rounds of loads. 182,640 rows, 20 columns: 12.5 us with one round per entry -> 6 us.
__global__ __launch_bounds__(kDotWaves * kLanes) void gm_dots_kernel(int64_t n, const double* __restrict__ V, int ncol,
                                                                     const double* __restrict__ w,
                                                                     double* __restrict__ part, int64_t nch) {
  __shared__ double row[kDotWaves][kLanes];
  const int wave = threadIdx.x / kLanes, l = threadIdx.x % kLanes;
  const int col = static_cast<int>(blockIdx.y) * kDotWaves + wave;
  if (col >= ncol) return;  // the whole wave
  const int64_t begin = static_cast<int64_t>(blockIdx.x) * kChunk;
  const int len = static_cast<int>(n - begin < kChunk ? n - begin : kChunk);
  const double t = wave_chunk_dot(V + col * n + begin, w + begin, len, l, row[wave]);
  if (l == 0) part[col * nch + blockIdx.x] = t;
}

// One workgroup per column: its chunk partials reduced level by level (more than kInlineParts).
__global__ __launch_bounds__(kLanes) void gm_totals_kernel(int64_t npart, const double* __restrict__ part,
                                                           double* __restrict__ out) {
  __shared__ double row[kLanes];
  __shared__ double tot[kChunk];
  const int l = threadIdx.x;
  const double* p = part + blockIdx.x * npart;
  const int64_t nch = chunks(npart);
  for (int64_t c = 0; c < nch; ++c) {
    const int64_t begin = c * kChunk;
    const double t = wave_chunk_sum(p, 1, begin, npart - begin < kChunk ? npart - begin : kChunk, l, row);
    if (l == 0) tot[c] = t;
  }
  __syncthreads();
  const double t = nch > 1 ? wave_chunk_sum(tot, 1, 0, nch, l, row) : tot[0];
  if (l == 0) out[blockIdx.x] = t;
}

// w -= sum_c h_c V(:, c) with h the totals of `dots` (the first workgroup keeps them in h), then the
// chunk partials of the next dots from the updated chunk: NEXT the second pass' V(:, c) . w, else
// w . w. One workgroup of eight waves per chunk; the chunk's columns come from L2 the second time.
constexpr int kOrthoWaves = 8;
template <bool NEXT>
__global__ __launch_bounds__(kOrthoWaves * kLanes) void gm_ortho_kernel(int64_t n, const double* __restrict__ V, int ncol,
                                                                        Dots dots, double* __restrict__ h,
                                                                        double* __restrict__ w,
                                                                        double* __restrict__ part, int64_t nch) {
  constexpr int NT = kOrthoWaves * kLanes, PER = kChunk / NT;
  __shared__ double ws[kChunk];
  __shared__ double row[kOrthoWaves][kLanes];
  __shared__ double coef[kGmresRestart + 1];
  const int t = threadIdx.x, wave = t / kLanes, l = t % kLanes;
  const int64_t begin = static_cast<int64_t>(blockIdx.x) * kChunk;
  const int len = static_cast<int>(n - begin < kChunk ? n - begin : kChunk);
  double wv[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int k = t + j * NT;
    wv[j] = w[begin + (k < len ? k : 0)];
  }
  for (int c = wave; c < ncol; c += kOrthoWaves) {
    const double s = wave_total(dots.part + c * dots.stride, 1, 0, dots.npart, l, row[wave]);
    if (l == 0) {
      coef[c] = -1.0 * s;
      if (blockIdx.x == 0) h[c] = s;
    }
  }
  __syncthreads();
  double s[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) s[j] = 0.0;
#pragma unroll 4
  for (int c = 0; c < ncol; ++c) {
    const double f = coef[c];
    const double* v = V + c * n + begin;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int k = t + j * NT;
      s[j] += f * v[k < len ? k : 0];
    }
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int k = t + j * NT;
    wv[j] += s[j];
    ws[k] = wv[j];
    if (k < len) w[begin + k] = wv[j];
  }
  __syncthreads();
  if constexpr (NEXT) {
    for (int c = wave; c < ncol; c += kOrthoWaves) {
      const double d = wave_chunk_dot(V + c * n + begin, ws, len, l, row[wave]);
      if (l == 0) part[c * nch + blockIdx.x] = d;
    }
  } else if (wave == 0) {
    const double d = wave_staged_dot(ws, ws, len, l, row[0]);
    if (l == 0) part[blockIdx.x] = d;
  }
}

// ||w|| from its chunk partials; v = w / ||w|| (as 0 + s w: VectorOps::fill then axpy) and z = inv v.
// The first workgroup writes the Hessenberg column h + h2, ||w|| to the host (hcol, ncol + 1
// entries), then the count of columns written.
__global__ __launch_bounds__(kVecThreads) void gm_next_kernel(int64_t n, const double* __restrict__ w, Dots norm,
                                                              const double* __restrict__ inv, double* __restrict__ v,
                                                              double* __restrict__ z, int ncol,
                                                              const double* __restrict__ h,
                                                              const double* __restrict__ h2, double* hcol, int32_t* ready) {
  __shared__ double row[kLanes];
  __shared__ double total;
  const int t = threadIdx.x;
  const int64_t begin = static_cast<int64_t>(blockIdx.x) * kChunk;
  const int len = static_cast<int>(n - begin < kChunk ? n - begin : kChunk);
  double wv[kPerThread], iv[kPerThread];
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    const int k = t + j * kVecThreads;
    wv[j] = w[begin + (k < len ? k : 0)];
    iv[j] = inv[begin + (k < len ? k : 0)];
  }
  if (t < kLanes) {
    const double s = wave_total(norm.part, 1, 0, norm.npart, t, row);
    if (t == 0) total = s;
  }
  __syncthreads();
  const double hn = sqrt(total), s = 1.0 / hn;
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    const int k = t + j * kVecThreads;
    const double vj = 0.0 + s * wv[j];
    if (k < len) {
      v[begin + k] = vj;
      z[begin + k] = iv[j] * vj;
    }
  }
  if (blockIdx.x == 0 && t == 0 && hcol) {
    for (int c = 0; c < ncol; ++c) hcol[c] = h[c] + h2[c];
    hcol[ncol] = hn;
    __hip_atomic_store(ready, ncol, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}
// w(i) += sum_c coef(c) V(i, c), V column-major with stride n
__global__ void gm_combine_kernel(int64_t n, int k, const double* __restrict__ coef, const double* __restrict__ V,
                                  double* __restrict__ w) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s = 0.0;
  for (int c = 0; c < k; ++c) s += coef[c] * V[c * n + i];
  w[i] += s;
}

}  // namespace

int gmres64_solver(fx_batch* b, const fx_coeffs& k, const fx_solve_options& o, const double* bi, double* xi,
                   fx_solve_result& res) {
  fx_ctx* ctx = b->ctx;
  hipStream_t st = ctx->stream;
  const int64_t n = b->neq;
  const int m = kGmresRestart;
  if (!b->gm) {
    ctx->error = "gmres: the batch was created without FX_BATCH_GMRES";
    return FX_EUNSUP;
  }
  double *w = b->work, *r = b->work + n, *inv = b->work + 4 * n, *d = b->work + 5 * n;
  const int64_t nch = chunks(n);
  double *V = b->gm, *Z = b->gm + (m + 1) * n;
  double* scratch = b->gm + (2 * m + 3) * n;
  double *part1 = scratch, *part2 = part1 + (m + 1) * nch, *tot = part2 + (m + 1) * nch, *hd = tot + m + 1,
         *hd2 = hd + m + 1, *coef = hd2 + m + 1;
  if (int rc = jacobi_inverse_public(b, k, d, inv)) return rc;
  res = fx_solve_result{};
  auto dot = [&](const double* x, const double* y, double& out) { return dot64(ctx, n, x, y, &out); };
  double bb = 0.0;
  if (int rc = dot(bi, bi, bb)) return rc;
  res.rhs_norm = std::sqrt(bb);
  const double tol = std::max(o.relative_tolerance * res.rhs_norm, o.absolute_tolerance);
  std::vector<double> H(static_cast<size_t>((m + 1) * m), 0.0), cs(m), sn(m), g(m + 1), y(m + 1);
  auto Hij = [&](int i, int j) -> double& { return H[static_cast<size_t>(j) * (m + 1) + i]; };
  // out += sum_c c_c base(:, c)
  auto combine = [&](const double* base, int kk, const std::vector<double>& c, double* out) -> int {
    FX_HIP(ctx, hipMemcpyAsync(coef, c.data(), sizeof(double) * kk, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(gm_combine_kernel, grid(n), dim3(kThreads), 0, st, n, kk, coef, base, out);
    FX_HIP(ctx, hipGetLastError());
    return FX_OK;
  };
  const dim3 per_chunk(static_cast<unsigned>(nch));
  auto dots_of = [&](const double* part, int ncol) {
    if (nch <= kInlineParts) return Dots{part, nch, nch};
    hipLaunchKernelGGL(gm_totals_kernel, dim3(ncol), dim3(kLanes), 0, st, nch, part, tot);
    return Dots{tot, 1, 1};
  };
  // the device's Hessenberg columns and their count
  char* pinned = static_cast<char*>(ctx->host_pinned) + 512;
  int32_t* ready = reinterpret_cast<int32_t*>(pinned);
  double* hcols = reinterpret_cast<double*>(pinned + 64);
  // Arnoldi step j: w = A z_j, two Gram-Schmidt passes (CGS2: one block of dots, one block update
  // each), the next basis vector and its preconditioned direction
  auto arnoldi = [&](int j) -> int {
    const int nc = j + 1;
    if (int rc = operator_apply64(b, k, Z + static_cast<size_t>(j) * n, w)) return rc;
    hipLaunchKernelGGL(gm_dots_kernel, dim3(per_chunk.x, (nc + kDotWaves - 1) / kDotWaves), dim3(kDotWaves * kLanes), 0,
                       st, n, V, nc, w, part1, nch);
    const Dots d1 = dots_of(part1, nc);
    hipLaunchKernelGGL(gm_ortho_kernel<true>, per_chunk, dim3(kOrthoWaves * kLanes), 0, st, n, V, nc, d1, hd, w, part2,
                       nch);
    const Dots d2 = dots_of(part2, nc);
    hipLaunchKernelGGL(gm_ortho_kernel<false>, per_chunk, dim3(kOrthoWaves * kLanes), 0, st, n, V, nc, d2, hd2, w, part1,
                       nch);
    const Dots nn = dots_of(part1, 1);
    // (the last step's z has no use; the workspace has a vector behind Z)
    hipLaunchKernelGGL(gm_next_kernel, per_chunk, dim3(kVecThreads), 0, st, n, w, nn, inv,
                       V + static_cast<size_t>(j + 1) * n, Z + static_cast<size_t>(j + 1) * n, nc, hd, hd2, hcols + static_cast<size_t>(j) * (m + 1), ready);
    FX_HIP(ctx, hipGetLastError());
    return FX_OK;
  };
  // until the device has written `cols` columns
  auto wait = [&](int cols) -> int {
    for (DeviceWait look; __atomic_load_n(ready, __ATOMIC_ACQUIRE) < cols;) {
      if (!look.pause()) continue;
      const hipError_t q = hipStreamQuery(st);
      if (q == hipErrorNotReady) continue;
      FX_HIP(ctx, q);
      if (__atomic_load_n(ready, __ATOMIC_ACQUIRE) < cols) {
        ctx->error = "GMRES: the device did not report the queued steps";
        return FX_EDEVICE;
      }
    }
    return FX_OK;
  };
  constexpr int kAhead = 3;  // Arnoldi steps queued beyond the one the host waits for
  bool first = true;
  for (;;) {
    if (int rc = operator_apply64(b, k, xi, w)) return rc;
    hipLaunchKernelGGL(gm_residual_kernel, grid(n), dim3(kThreads), 0, st, n, bi, w, r);
    double rr = 0.0;
    if (int rc = dot(r, r, rr)) return rc;
    const double beta = std::sqrt(rr);
    if (first) res.initial_residual = beta;
    first = false;
    res.final_residual = beta;
    if (beta <= tol) {
      res.converged = 1;
      return FX_OK;
    }
    if (res.iterations >= o.max_iterations) return FX_OK;
    __atomic_store_n(ready, 0, __ATOMIC_RELEASE);
    // V(:, 0) = r / beta and z_0: beta^2 is the residual's dot, summed again from its chunk partials
    hipLaunchKernelGGL(gm_dots_kernel, dim3(per_chunk.x, 1), dim3(kDotWaves * kLanes), 0, st, n, r, 1, r, part1, nch);
    const Dots rd = dots_of(part1, 1);
    hipLaunchKernelGGL(gm_next_kernel, per_chunk, dim3(kVecThreads), 0, st, n, r, rd, inv, V, Z, 0, hd, hd2,
                       static_cast<double*>(nullptr), ready);
    std::fill(g.begin(), g.end(), 0.0);
    g[0] = beta;
    const int steps = std::min(m, o.max_iterations - res.iterations);
    int j = 0, queued = 0;
    while (j < steps) {
      for (; queued < steps && queued <= j + kAhead; ++queued)
        if (int rc = arnoldi(queued)) return rc;
      if (int rc = wait(j + 1)) return rc;
      const double* col = hcols + static_cast<size_t>(j) * (m + 1);
      for (int i = 0; i <= j; ++i) Hij(i, j) = col[i];
      const double hn = col[j + 1];
      for (int i = 0; i < j; ++i) {
        const double a = Hij(i, j), c = Hij(i + 1, j);
        Hij(i, j) = cs[i] * a + sn[i] * c;
        Hij(i + 1, j) = -sn[i] * a + cs[i] * c;
      }
      const double a = Hij(j, j), c = hn;
      const double dd = std::hypot(a, c);
      cs[j] = dd > 0.0 ? a / dd : 1.0;
      sn[j] = dd > 0.0 ? c / dd : 0.0;
      Hij(j, j) = dd;
      Hij(j + 1, j) = 0.0;
      g[j + 1] = -sn[j] * g[j];
      g[j] = cs[j] * g[j];
      ++res.iterations;
      ++j;
      res.final_residual = std::fabs(g[j]);
      if (res.final_residual <= tol || hn == 0.0) break;
    }
    for (int i = j - 1; i >= 0; --i) {
      double s = g[i];
      for (int kk = i + 1; kk < j; ++kk) s -= Hij(i, kk) * y[kk];
      y[i] = s / Hij(i, i);
    }
    if (int rc = combine(Z, j, y, xi)) return rc;
    if (res.final_residual <= tol) {
      if (int rc = operator_apply64(b, k, xi, w)) return rc;
      hipLaunchKernelGGL(gm_residual_kernel, grid(n), dim3(kThreads), 0, st, n, bi, w, r);
      double r2 = 0.0;
      if (int rc = dot(r, r, r2)) return rc;
      res.final_residual = std::sqrt(r2);
      if (res.final_residual <= tol) {
        res.converged = 1;
        return FX_OK;
      }
    }
    if (res.iterations >= o.max_iterations) return FX_OK;
  }
}

int krylov64_solver(fx_batch* b, const fx_coeffs& k, const fx_solve_options& o, const double* bi, double* xi,
                    fx_solve_result& res) {
  const int64_t n = b->neq;
  if (!operator_spd(b, k)) {  // KrylovSolver::setup (krylov.cpp:10-22): GMRES from the start
    if (!b->gm) {
      b->ctx->error = "Krylov solve: the operator is not symmetric positive definite, so it needs GMRES (create "
                      "the batch with FX_BATCH_GMRES)";
      return FX_EINVAL;
    }
    res = fx_solve_result{};
    return gmres64_solver(b, k, o, bi, xi, res);
  }
  double* x0 = b->gm ? b->gm + (2 * kGmresRestart + 2) * n : nullptr;
  if (x0)
    if (int rc = copy64(b->ctx, n, xi, x0)) return rc;
  if (int rc = cg64_solver(b, k, o, bi, xi, res)) return rc;
  if (!res.indefinite || !x0) return FX_OK;
  const int cg_iterations = res.iterations;
  if (int rc = copy64(b->ctx, n, x0, xi)) return rc;
  if (int rc = gmres64_solver(b, k, o, bi, xi, res)) return rc;
  res.iterations += cg_iterations;
  res.indefinite = 1;
  return FX_OK;
}

}  // namespace fx
